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
    for (size_t n : {4ul, 36ul, 350000ul, MiB, MiB + 4, 4 * MiB / 3, 4 * MiB / 3 / 4 * 4 + 4, 2 * MiB - 4, 2 * MiB + 8, 7 * MiB + 12, 11 * MiB})
        for (bool skip : {false, true}) reads(st, &s, n, skip);
    reads(st, &s, 4, false);
}

// A readback of one chunk makes one copy and one wait, no event: what the
// runtime's own copy costs a small frame.
static void one_chunk()
{
    fake::Stream s;
    Staging st;
    for (size_t n : {8ul, 40000ul, MiB / 3}) {
        fake::waits = fake::records = 0;
        reads(st, &s, n, false);
        CHECK(fake::waits == 1 && fake::records == 0);
    }
    fake::waits = fake::records = 0;
    reads(st, &s, MiB, false);  // three chunks
    CHECK(fake::waits == 3 && fake::records == 2);
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
    for (size_t n : {MiB, 2 * MiB, 11 * MiB})
        for (int left : {0, 1, 2}) {
            fake::copies_left = left;
            reads(st, &s, n, false, hipErrorUnknown);
            fake::copies_left = -1;
            reads(st, &s, n, false);
        }
}

// Pinned memory does not grow with the objects, is given back with the last of
// them, and is not taken before a readback asks for it.
static void pinned()
{
    fake::Stream s;
    CHECK(fake::pinned == 0);
    for (int round = 0; round < 2; ++round) {
        std::vector<std::unique_ptr<Staging>> many;
        for (int k = 0; k < 200; ++k) many.push_back(std::make_unique<Staging>());
        CHECK(fake::pinned == 0 && fake::events == 0);
        reads(*many[0], &s, 1000, false);
        CHECK(fake::pinned <= MiB);
        for (auto& st : many) reads(*st, &s, 100000, false);
        CHECK(fake::pinned <= 2 * MiB);
        reads(*many[3], &s, 11 * MiB, false);
        reads(*many[4], &s, 11 * MiB, false);
        CHECK(fake::pinned <= 12 * MiB);
        while (many.size() > 1) many.pop_back();
        reads(*many[0], &s, 3 * MiB, true);
        many.clear();
        CHECK(fake::pinned == 0 && fake::events == 0);
    }
    CHECK(fake::pinned_most <= 12 * MiB);
}

// Objects of their own on streams of their own, each driven by one thread, at
// the same time; one is made and ended again and again.
static void together()
{
    std::vector<std::thread> threads;
    for (int t = 0; t < 5; ++t)
        threads.emplace_back([t] {
            fake::Stream s;
            std::unique_ptr<Staging> st = std::make_unique<Staging>();
            for (int k = 0; k < 12; ++k) {
                const size_t n = (size_t)(1 + (t * 7 + k * 5) % 13) * MiB + 4 * t;
                std::vector<unsigned> src = device(n, (unsigned)(t + k));
                std::vector<char> out(n + 1, 77);
                const HostPiece p{out.data(), src.data(), n};
                CHECK(st->to_host(&p, 1, &s, t == 4 ? 64 : 0) == hipSuccess);
                CHECK(std::memcmp(out.data(), src.data(), n) == 0 && out[n] == 77);
                if (t == 0) st = std::make_unique<Staging>();
            }
        });
    for (std::thread& t : threads) t.join();
    CHECK(fake::pinned_most <= 12 * MiB);
    CHECK(fake::pinned == 0 && fake::events == 0);
}

// Without pinned memory or events the readback goes the runtime's way; with
// some of them it takes what there is.
static void short_of_memory()
{
    fake::Stream s;
    for (size_t n : {1000ul, MiB, 2 * MiB})
        for (int good : {0, 1, 5}) {
            Staging st;
            if (good) reads(st, &s, (good == 1 ? 1 : 4) * MiB / 4, false);
            fake::fail_pin = 1000;
            reads(st, &s, n, false);
            fake::fail_pin = 0;
            fake::fail_event = 1;
            reads(st, &s, n, true);
            fake::fail_event = 0;
            reads(st, &s, n, false);
        }
    CHECK(fake::pinned == 0 && fake::events == 0);
}

int main(int argc, char** argv)
{
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "bytes") bytes();
    else if (what == "one_chunk") one_chunk();
    else if (what == "busy") busy();
    else if (what == "copy_fails") copy_fails();
    else if (what == "pinned") pinned();
    else if (what == "together") together();
    else if (what == "short_of_memory") short_of_memory();
    else return 2;
    std::printf("%s ok\n", what.c_str());
    return 0;
}
