// k3_step2 (lbm3d.hip) run on the CPU, block by block, against two passes of
// the same source's one-step cell3: the same bits at every slot a fluid cell
// can read and no write anywhere else, with the threads in either order between
// barriers.  LDS is one static block that keeps what the block before left.
#include <cstdio>
#include <cstring>
#include <random>

#include "lbm3d_kernels.hpp"

using namespace lbm;
using namespace lbm::d3;

static emu::Block g_block;

template <typename T, bool FORCE, int BS, int RW>
static bool one_case(int nx, int ny, int nz, int depth, bool backwards)
{
    constexpr int RH = BS / RW;
    Args3 a{};
    a.nx = nx;
    a.ny = ny;
    a.nz = nz;
    a.pitch = ((uint32_t)nx + 15u) & ~15u;
    a.rs = 19u * a.pitch;
    a.omega = 1.0f / 0.7f;
    a.gx = FORCE ? 2e-5f : 0.0f;
    a.gy = FORCE ? -1e-5f : 0.0f;
    a.gz = FORCE ? 3e-5f : 0.0f;
    a.scale = 1024.0f;
    a.inv_scale = 1.0f / 1024.0f;
    set_force_terms3(a);
    const int rows = ny * nz;
    const size_t elems = (size_t)a.rs * rows;
    std::mt19937 rng(nx * 131 + ny * 17 + nz);
    std::vector<uint8_t> solid((size_t)nx * rows);
    for (auto& s : solid) s = rng() % 14 == 0;
    solid[0] = solid.back() = 1;
    const uint32_t words = solid_mask_words(nx);
    std::unique_ptr<uint32_t[]> bits(new uint32_t[(size_t)words * rows]());
    for (int r = 0; r < rows; ++r)
        for (uint32_t b = 0; b < (uint32_t)nx + 2; ++b)
            if (solid[(size_t)r * nx + ((int)b - 1 + nx) % nx]) bits[(size_t)r * words + b / 32] |= 1u << (b % 32);
    const auto at = [&](int x, int y, int z, int i) {
        return ((size_t)((z + nz) % nz) * ny + (y + ny) % ny) * a.rs + (size_t)i * a.pitch + (x + nx) % nx;
    };
    const auto is_solid = [&](int x, int y, int z) {
        return solid[((size_t)((z + nz) % nz) * ny + (y + ny) % ny) * nx + (x + nx) % nx] != 0;
    };
    std::vector<char> seen(elems, 0);
    std::unique_ptr<T[]> src(new T[elems]), mid(new T[elems]), want(new T[elems]), dst(new T[elems]);
    std::uniform_real_distribution<float> u(-1.0f, 1.0f);
    const float size = sizeof(T) == 2 ? 4.0f : 4e-3f, mark = sizeof(T) == 2 ? 777.0f : 0.777f;
    for (size_t k = 0; k < elems; ++k) src[k] = (T)(size * u(rng));
    for (int z = 0; z < nz; ++z)
        for (int y = 0; y < ny; ++y)
            for (int x = 0; x < nx; ++x)
                for (int i = 0; i < 19; ++i) {
                    const int tx = x + ex3(i), ty = y + ey3(i), tz = z + ez3(i);
                    const bool s = is_solid(x, y, z), pulls = i > 0 && !is_solid(tx, ty, tz);
                    if (!s || pulls) seen[at(x, y, z, i)] = 1;
                    if (s && pulls) src[at(x, y, z, i)] = src[at(tx, ty, tz, inv3(i))];
                }
    std::memcpy(mid.get(), src.get(), elems * sizeof(T));
    std::memcpy(want.get(), src.get(), elems * sizeof(T));
    for (int step = 0; step < 2; ++step)
        for (int z = 0; z < nz; ++z)
            for (int y = 0; y < ny; ++y)
                for (int x = 0; x < nx; ++x)
                    cell3<T, FORCE, 0>(a, step ? mid.get() : src.get(), step ? want.get() : mid.get(), bits.get(), words, x, y, z);
    for (size_t k = 0; k < elems; ++k) dst[k] = (T)mark;
    const uint32_t tx = (uint32_t)((nx + RW - 3) / (RW - 2)), ty = (uint32_t)((ny + RH - 3) / (RH - 2));
    const uint32_t tz = (uint32_t)((nz + depth - 1) / depth);
    gridDim.x = tx * ty * tz;
    for (blockIdx.x = 0; blockIdx.x < gridDim.x; ++blockIdx.x)
        if (!g_block.run(BS, backwards, [&] {
                k3_step2<T, FORCE, BS, RW, 0>(a, src.get(), dst.get(), bits.get(), words, tx, ty, depth);
            })) {
            std::printf("barriers differ between threads\n");
            return false;
        }
    size_t wrong = 0, stray = 0;
    for (size_t k = 0; k < elems; ++k) {
        if (seen[k]) wrong += std::memcmp(&dst[k], &want[k], sizeof(T)) != 0;
        else stray += (float)dst[k] != (float)(T)mark;
    }
    if (wrong || stray)
        std::printf("%s force %d block %d width %d lattice %dx%dx%d depth %d backwards %d: %zu slots differ, %zu stray writes\n",
                    sizeof(T) == 2 ? "f16" : "f32", FORCE, BS, RW, nx, ny, nz, depth, backwards, wrong, stray);
    return wrong + stray == 0;
}

template <int BS, int RW>
static int shape()
{
    constexpr int W = RW - 2, H = BS / RW - 2;
    // nx, ny, nz, slabs of a chunk: the smallest; whole tiles; one column and
    // row more and a last chunk of one slab
    const int sizes[][4] = {{3, 3, 3, 3}, {3, 3, 3, 1}, {W, H, 4, 2}, {W + 1, H + 1, 5, 2}, {W - 1, 2 * H + 1, 4, 3}};
    int bad = 0;
    for (const auto& s : sizes)
        for (bool backwards : {false, true}) {
            bad += !one_case<float, false, BS, RW>(s[0], s[1], s[2], s[3], backwards);
            bad += !one_case<float, true, BS, RW>(s[0], s[1], s[2], s[3], backwards);
            bad += !one_case<_Float16, true, BS, RW>(s[0], s[1], s[2], s[3], backwards);
        }
    return bad;
}

int main()
{
    const int bad = shape<512, 64>() + shape<1024, 32>();
    std::printf("two steps: %d bad\n", bad);
    return bad != 0;
}
