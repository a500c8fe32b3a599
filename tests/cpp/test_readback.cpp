// lbm_readback.hpp against a stand-in runtime (fake_hip): the bytes of every
// split, who waits while the stream is busy, how much memory stays pinned, and
// what happens where an allocation or a copy fails.
#include <chrono>
#include <cstdio>
#include <memory>
#include <string>
#include <vector>

#include "lbm_readback.hpp"

using lbm::HostPiece;
using lbm::Staging;

#define CHECK(c)                                                          \
    do {                                                                  \
        if (!(c)) {                                                       \
            std::printf("line %d: %s does not hold\n", __LINE__, #c);     \
            std::exit(1);                                                 \
        }                                                                 \
    } while (0)

static constexpr size_t MiB = 1u << 20;

static std::vector<unsigned> device(size_t bytes, unsigned salt)
{
    std::vector<unsigned> v(bytes / 4 + 1);
    for (size_t k = 0; k < v.size(); ++k) v[k] = (unsigned)k * 2654435761u + salt;
    return v;
}

// Three pieces of `bytes`, one behind the other on the device; the second one
// skipped with `skip`.
static void reads(Staging& st, hipStream_t s, size_t bytes, bool skip, hipError_t want = hipSuccess)
{
    const std::vector<unsigned> src = device(3 * bytes, (unsigned)bytes);
    const char* const from = (const char*)src.data();
    std::vector<char> out[3];
    HostPiece p[3];
    for (int k = 0; k < 3; ++k) {
        out[k].assign(bytes + 1, 77);
        p[k] = {skip && k == 1 ? nullptr : out[k].data(), from + k * bytes, bytes};
    }
    const hipError_t e = st.to_host(p, 3, s, 0);
    CHECK(e == want);
    CHECK(fake::waiting == 0);
    s->drain();  // nothing may be left that reads src or writes a slot
    if (want != hipSuccess) return;
    for (int k = 0; k < 3; ++k) {
        if (skip && k == 1) continue;
        CHECK(std::memcmp(out[k].data(), from + k * bytes, bytes) == 0);
        CHECK(out[k][bytes] == 77);
    }
}

static void bytes()
{
    fake::Stream s;
    Staging st;
    for (size_t n : {4ul, 36ul, 350000ul, MiB, MiB + 4, 2 * MiB - 4, 2 * MiB + 8, 7 * MiB + 12, 11 * MiB, 17 * MiB})
        for (bool skip : {false, true}) reads(st, &s, n, skip);
    reads(st, &s, 4, false);
}

// While the stream has other work before the readback, only the calling thread
// waits inside the runtime, whose waits spin.
static void busy()
{
    fake::Stream s;
    Staging st;
    s.hold(true);
    s.push([] {});
    std::thread caller([&] { reads(st, &s, 14 * MiB, false); });
    int most = 0;
    while (fake::waiting == 0) std::this_thread::sleep_for(std::chrono::milliseconds(1));
    for (int k = 0; k < 200; ++k) {
        most = std::max(most, fake::waiting.load());
        std::this_thread::sleep_for(std::chrono::milliseconds(1));
    }
    s.hold(false);
    caller.join();
    CHECK(most == 1);
}

// A failing copy ends the readback with its error, every thread ended and
// nothing in flight; the next readback is whole again.
static void copy_fails()
{
    fake::Stream s;
    Staging st;
    for (size_t n : {MiB, 3 * MiB, 14 * MiB})
        for (int left : {0, 1, 2}) {
            fake::copies_left = left;
            reads(st, &s, n, false, hipErrorUnknown);
            fake::copies_left = -1;
            reads(st, &s, n, false);
        }
}

int main(int argc, char** argv)
{
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "bytes") bytes();
    else if (what == "busy") busy();
    else if (what == "copy_fails") copy_fails();
    else return 2;
    std::printf("%s ok\n", what.c_str());
    return 0;
}
