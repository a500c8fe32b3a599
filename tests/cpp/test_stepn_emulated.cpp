// The body of the N-step tile kernels (lbm_stepn.hip) run on the CPU, tile by
// tile, against as many one-step passes of the same source's phys_cell: the
// same bits at every slot a fluid cell can read and no write anywhere else,
// whatever lies in LDS before, in whatever order the threads come between
// barriers, and with either answer of __any.  Populations, mask and LDS are
// heap blocks of their exact size, so the address sanitizer sees a read or
// write beyond them, and the bounds sanitizer one beyond an LDS plane.
#include <cstdio>
#include <cstring>
#include <random>
#include <string>

#include "lbm_stepn_tile.hpp"

using namespace lbm;

bool lbm::two_step_fits(int bw, int nx, int ny, int xedge) { return nx >= 3 && ny >= 3 && (xedge == 0 || nx % bw != 1); }

static emu::Block g_block;

template <typename T, int XEDGE, bool FORCE, int RW, int RH, int NS>
static bool one_case(int nx, int ny, bool planes, int flavour)
{
    constexpr int BS = 1024, BW = RW - 2 * (NS - 1), BH = RH - 2 * (NS - 1);
    if (!nstep_fits(BW, NS, nx, ny, XEDGE)) return true;
    PhysArgs a{};
    a.nx = nx;
    a.ny = ny;
    const uint32_t n = (uint32_t)nx * (uint32_t)ny, pitch = ((uint32_t)nx + 15u) & ~15u;
    a.plane = planes ? (n + 63u) & ~63u : pitch;
    a.rs = planes ? (uint32_t)nx : 9u * pitch;
    const size_t elems = planes ? (size_t)9 * a.plane : (size_t)a.rs * ny;
    a.omega = 1.0f / 0.7f;
    a.gx = FORCE ? 2e-5f : 0.0f;
    a.gy = FORCE ? -1e-5f : 0.0f;
    a.inlet_ux = XEDGE ? 0.04f : 0.0f;
    a.scale = 1024.0f;
    a.inv_scale = 1.0f / 1024.0f;
    set_force_terms(a);
    std::mt19937 rng(nx * 131 + ny);
    std::vector<uint8_t> solid(n);
    for (int y = 0; y < ny; ++y)
        for (int x = 0; x < nx; ++x)
            solid[(size_t)y * nx + x] = (XEDGE && (y == 0 || y == ny - 1)) || rng() % 16 == 0 ||
                                        (XEDGE && x >= nx - 2 && y % 7 == 3) || (x < 2 && y % 9 == 4);
    const uint32_t words = solid_mask_words(nx);
    std::unique_ptr<uint32_t[]> bits(new uint32_t[(size_t)words * ny]());
    for (int y = 0; y < ny; ++y)
        for (uint32_t b = 0; b < 32 * words; ++b) {
            int x = (int)b - 1;
            if (x > nx || (XEDGE && (x < 0 || x == nx))) continue;
            x = x < 0 ? nx - 1 : (x == nx ? 0 : x);
            if (solid[(size_t)y * nx + x]) bits[(size_t)y * words + b / 32] |= 1u << (b % 32);
        }
    const auto at = [&](int x, int y, int i) { return (size_t)y * a.rs + (size_t)x + (size_t)i * a.plane; };
    std::vector<char> seen(elems, 0);  // slots a fluid cell can read, of the destination
    for (int y = 0; y < ny; ++y)
        for (int x = 0; x < nx; ++x)
            for (int i = 0; i < 9; ++i) {
                const int tx = x + ex_of(i), ty = (y + ey_of(i) + ny) % ny;
                const bool inside = tx >= 0 && tx < nx;
                const bool pulls = (inside || !XEDGE) && !solid[(size_t)ty * nx + (tx + nx) % nx];
                if (!solid[(size_t)y * nx + x] || (i > 0 && pulls)) seen[at(x, y, i)] = 1;
            }
    std::unique_ptr<T[]> src(new T[elems]), dst(new T[elems]), one[2] = {std::unique_ptr<T[]>(new T[elems]), std::unique_ptr<T[]>(new T[elems])};
    std::uniform_real_distribution<float> u(-1.0f, 1.0f);
    const float size = sizeof(T) == 2 ? 4.0f : 4e-3f, mark = sizeof(T) == 2 ? 777.0f : 0.777f;
    for (size_t k = 0; k < elems; ++k) src[k] = (T)(size * u(rng));
    // what a pull from a solid cell finds: the fluid neighbour's own opposite
    for (int y = 0; y < ny; ++y)
        for (int x = 0; x < nx; ++x)
            for (int i = 1; i < 9; ++i) {
                const int tx = x + ex_of(i), ty = (y + ey_of(i) + ny) % ny;
                if (!solid[(size_t)y * nx + x] || (XEDGE && (tx < 0 || tx >= nx))) continue;
                const int wx = (tx + nx) % nx;
                if (!solid[(size_t)ty * nx + wx]) src[at(x, y, i)] = src[at(wx, ty, inv_of(i))];
            }
    std::memcpy(one[0].get(), src.get(), elems * sizeof(T));
    std::memcpy(one[1].get(), src.get(), elems * sizeof(T));
    for (int s = 0; s < NS; ++s)
        for (int y = 0; y < ny; ++y)
            for (int x = 0; x < nx; ++x)
                phys_cell<T, XEDGE, FORCE, false>(a, one[s & 1].get(), one[(s & 1) ^ 1].get(), bits.get(), words, nullptr, n, x, y);
    const T* const want = one[NS & 1].get();
    for (size_t k = 0; k < elems; ++k) dst[k] = (T)mark;
    const std::unique_ptr<T[][RW * RH]> lds(new T[9][RW * RH]);
    const float poison[2] = {NAN, sizeof(T) == 2 ? -6e4f : 3e38f};
    emu::any_mode = flavour & 1;
    for (int y0 = 0; y0 < ny; y0 += BH)
        for (int x0 = 0; x0 < nx; x0 += BW) {
            for (int i = 0; i < 9; ++i)
                for (int c = 0; c < RW * RH; ++c) lds[i][c] = (T)poison[flavour & 1];
            const bool ok = g_block.run(BS, flavour & 2, [&] {
                nstep_tile<T, XEDGE, FORCE, BS, RW, RH, NS, 0>(a, src.get(), dst.get(), bits.get(), words, x0, y0, lds.get());
            });
            if (!ok) {
                std::printf("barriers differ between threads\n");
                return false;
            }
        }
    size_t wrong = 0, stray = 0;
    for (size_t k = 0; k < elems; ++k) {
        if (seen[k]) wrong += std::memcmp(&dst[k], &want[k], sizeof(T)) != 0;
        else stray += (float)dst[k] != (float)(T)mark;
    }
    if (wrong || stray)
        std::printf("%s edge %d force %d region %dx%d steps %d lattice %dx%d planes %d flavour %d: %zu slots differ, %zu stray writes\n",
                    sizeof(T) == 2 ? "f16" : "f32", XEDGE, FORCE, RW, RH, NS, nx, ny, planes, flavour, wrong, stray);
    return wrong + stray == 0;
}

template <typename T, int RW, int RH, int NS>
static int shape()
{
    constexpr int BW = RW - 2 * (NS - 1), BH = RH - 2 * (NS - 1);
    // the smallest; the ring wrapped in both directions; one cell more than a
    // tile; a two-column last tile, cut in y; several tiles, uncut, and with the
    // second one's ring at the lattice's last cells and one short of them
    const int sizes[][2] = {{NS, NS}, {NS + 3, NS + 1}, {BW + 1, BH + 1}, {2 * BW + 2, BH - 3}, {3 * BW, 3 * BH},
                            {2 * BW + NS - 1, 2 * BH + NS}, {2 * BW + NS, 2 * BH + NS - 1}};
    int bad = 0, k = 0;
    for (const auto& s : sizes)
        for (int flavour : {0, 3}) {  // own predicates, forwards, NaN in LDS; always true, backwards, huge values
            const bool planes = ++k / 2 % 2;
            bad += !one_case<T, 0, false, RW, RH, NS>(s[0], s[1], planes, flavour);
            bad += !one_case<T, 0, true, RW, RH, NS>(s[0], s[1], !planes, flavour);
            bad += !one_case<T, 1, false, RW, RH, NS>(s[0], s[1], !planes, flavour);
            bad += !one_case<T, 1, true, RW, RH, NS>(s[0], s[1], planes, flavour);
        }
    return bad;
}

int main(int argc, char** argv)
{
    const std::string what = argc > 1 ? argv[1] : "";
    int bad;
    if (what == "32x32x9") bad = shape<float, 32, 32, 9>() + shape<_Float16, 32, 32, 9>();
    else if (what == "32x32x5") bad = shape<float, 32, 32, 5>() + shape<_Float16, 32, 32, 5>();
    else if (what == "64x32x5") bad = shape<float, 64, 32, 5>() + shape<_Float16, 64, 32, 5>();
    else if (what == "64x48x5") bad = shape<float, 64, 48, 5>() + shape<_Float16, 64, 48, 5>();
    else return 2;
    std::printf("%s: %d bad\n", what.c_str(), bad);
    return bad != 0;
}
