// lbm_stepn.hip -- N steps per launch for one domain (N = 3 .. 9), a region
// of power-of-two width in LDS with every thread bound to its cells for the
// whole launch; its launcher and shape table.
#include <type_traits>

#include "lbm_cell.hpp"
#include "lbm_device.hpp"
#include "lbm_internal.hpp"

namespace lbm {

// A block of BS threads owns a region of RW x RH cells, RW a power of two:
// a tile of (RW - 2 (NS - 1)) x (RH - 2 (NS - 1)) cells with a ring of
// NS - 1.  Thread t owns the region cells t + BS m.  Step 1 gathers the
// whole region from HBM into LDS, step s runs on the cells s - 1 in from
// the region's rim, from LDS into LDS, and step NS runs on the tile and
// stores to HBM with the pushes into solid neighbours.  The rules of a step
// are the three-step tile's: a population from a solid cell, or from outside
// the channel, is the gathering cell's own opposite one; column 0 applies
// the Zou-He inlet; the outlet column gathers as its west neighbour.  They
// depend on the cell alone, so each thread reads its cells' solid mask once
// and keeps the outcome in one word per cell.  The destination ends up as NS
// one-step launches leave it (at every slot a fluid cell can read); NS is
// odd, so also in the same buffer.
//
// What bounds it: in binary32 no unit alone.  At 4096^2 the SIMDs issue vector
// instructions for about half of a launch (binary32 arithmetic and 32-bit
// logic take two cycles of a SIMD, shifts, compares, selects and conversions
// four), the LDS is busy for 26 % without bank conflicts, HBM carries one read
// and one write of the state per NS steps (1.40 GB, 3.6 TB/s), and wavefronts
// wait for half of their time on the chain of loads, collision and barriers.
// In binary16 the conversions bring the issue to two thirds to three quarters.
// Fewer instructions shorten both the chain and the issue: with the masks read
// once, addresses that a step only reads with constant offsets and the step
// loop unrolled, a pass of 64 cells takes 83 of them in binary32 with force
// between LDS and LDS, where the three-step tile takes 128.  That is what makes
// the wider ring of five steps pay: 4096^2 binary32 periodic with force 72 us per step against 90
// for the three-step 64 x 24 tile, 8192^2 binary16 253 (64 x 48 region)
// against 281.  On small lattices the launches count instead (a launch of a
// few blocks takes about 3 us, however little it computes): 256^2 1.3 us per
// step with nine steps per launch against 3.8 with one.  A step loop left
// rolled keeps the registers of every step live and spills with two cells
// per thread (the build refuses that); seven steps on the 64 x 32 region lose more to the ring than
// they save (74 against 72 us), and binary32 regions of 64 x 48 leave one
// block per CU (95).
enum : uint32_t {
    kPullMask = 0x1FFu,    // solid flags a gather looks at: rows above, of the cell, below (x - 1, x, x + 1 each)
    kNearShift = 9,        // the same 9 flags of the cell itself, for the pushes
    kOutletBit = 1u << 18, // gathers as its west neighbour
    kInletBit = 1u << 19,  // Zou-He inlet column
    kLiveBit = 1u << 20,   // a fluid cell of the lattice
    kSlowMask = kPullMask | kOutletBit | kInletBit
};
// Bit of kPullMask that holds the source cell x - e_i of direction i.
constexpr int pull_bit(int i) { return (ey_of(i) == 1 ? 0 : (ey_of(i) == 0 ? 3 : 6)) + 1 - ex_of(i); }

// Solid flags (x - 1, x, x + 1) of a mask row: one funnel shift of the two
// words from p on.
__device__ __forceinline__ uint32_t mask3(const uint32_t* __restrict__ p, uint32_t x)
{
    return __builtin_amdgcn_alignbit(p[1], p[0], x & 31u) & 7u;
}

// a where bit `bit` of d is set, else b, as a merge under the sign-extended
// bit (two instructions; a plain select of two LDS values makes the compiler
// select their addresses instead).
template <typename T>
__device__ __forceinline__ T pick(uint32_t d, int bit, T a, T b)
{
    using U = std::conditional_t<sizeof(T) == 2, uint16_t, uint32_t>;
    uint32_t m = (uint32_t)__builtin_amdgcn_sbfe((int)d, bit, 1);
    asm volatile("" : "+v"(m));
    const uint32_t ua = __builtin_bit_cast(U, a), ub = __builtin_bit_cast(U, b);
    return __builtin_bit_cast(T, (U)((ua & m) | (ub & ~m)));
}

// Element `off` past the uniform `base`, at the lane's column x of the
// lattice row that `row` elements further begin.  Where a wavefront holds
// cells of one row (ROW) everything but x is uniform, so the address is a
// scalar base and a 32-bit lane offset; elsewhere one pointer per lane.
template <bool ROW, typename T>
__device__ __forceinline__ T* elem(T* base, uint32_t row, int x, ptrdiff_t off)
{
    using C = std::conditional_t<std::is_const_v<T>, const char, char>;
    if constexpr (ROW) return reinterpret_cast<T*>(reinterpret_cast<C*>(base + row + off) + (uint32_t)x * (uint32_t)sizeof(T));
    else return base + (row + (uint32_t)x) + off;
}

template <typename T, int XEDGE, bool FORCE, int BS, int RW, int RH, int NS, int FLAGS>
__device__ inline void nstep_tile(const PhysArgs& a_in, const T* __restrict__ src, T* __restrict__ dst,
                                  const uint32_t* __restrict__ bits, uint32_t words, int x0, int y0,
                                  T (*__restrict__ lds)[RW * RH])
{
    PhysArgs a = a_in;
    constexpr bool SC = kScaledDom<T>;
    if (FORCE) pin_pair_consts<SC>(a);
    constexpr int RC = RW * RH, CPT = RC / BS, RSTEP = BS / RW, RING = NS - 1;
    constexpr int BW = RW - 2 * RING, BH = RH - 2 * RING;
    constexpr bool kRowWave = RW % 64 == 0;  // a wavefront holds cells of one row
    static_assert(RC % BS == 0 && BS % RW == 0 && BW > 0 && BH > 0 && NS >= 2, "region and block");
    const int nx = a.nx, ny = a.ny;
    const int q = (int)threadIdx.x % RW;
    int rq = (int)threadIdx.x / RW;
    if constexpr (kRowWave) rq = __builtin_amdgcn_readfirstlane(rq);

    // Regions whose gathers stay inside the lattice need no wrap.
    const bool inner = x0 > RING && x0 + BW + RING < nx && y0 > RING && y0 + BH + RING < ny;
    const int xr = x0 - RING + q;  // unwrapped column, the same for all of a thread's cells
    uint32_t cell[CPT];

    // Step 1 and each cell's gather rule.
#pragma unroll
    for (int m = 0; m < CPT; ++m) {
        const int r = rq + RSTEP * m;
        int x = xr, y = y0 - RING + r;
        float g[9];
        uint32_t near;
        if (inner) {
            const uint32_t* const w = bits + (__umul24((uint32_t)y, words) + ((uint32_t)x >> 5));
            near = mask3(w - words, (uint32_t)x) | (mask3(w, (uint32_t)x) << 3) | (mask3(w + words, (uint32_t)x) << 6);
            const uint32_t row = __umul24((uint32_t)y, a.rs);
#pragma unroll
            for (int i = 0; i < 9; ++i) {
                const ptrdiff_t off = (ptrdiff_t)((uint32_t)i * a.plane) - (ptrdiff_t)ey_of(i) * (ptrdiff_t)a.rs -
                                      (ptrdiff_t)ex_of(i);
                g[i] = Dom<T, SC>::in(*elem<kRowWave>(src, row, x, off), a.inv_scale);
            }
            cell[m] = (near * (1u + (1u << kNearShift))) | ((near & 16u) ? 0u : kLiveBit);
        } else {
            cell[m] = 0u;
            // rim tiles: y in a vector register, the scalar ones are taken by the uniform addresses
            asm volatile("" : "+v"(y));
            // beyond the ring of a cut tile, or outside the channel: never read
            if (x >= nx + RING || y >= ny + RING) continue;
            if (XEDGE == 1 && (x < 0 || x >= nx)) continue;
            x = x < 0 ? x + nx : (x >= nx ? x - nx : x);
            y = y < 0 ? y + ny : (y >= ny ? y - ny : y);
            const CellNbr nb = cell_nbr(a, bits, words, x, y);
            cell_gather<T, XEDGE, 0, SC>(a, src, nb, x, y, g);
            near = nb.sm | (nb.s0 << 3) | (nb.sp << 6);
            uint32_t d = (near << kNearShift) | ((near & 16u) ? 0u : kLiveBit);
            if constexpr (XEDGE == 1) {
                int cx = x;
                if (x == nx - 1 && !(nb.s0 & 1u)) {
                    d |= kOutletBit;
                    cx = x - 1;
                    const CellNbr gb = cell_nbr(a, bits, words, cx, y);
                    near = gb.sm | (gb.s0 << 3) | (gb.sp << 6);
                }
                // sources outside the channel: the cell's own opposite
                if (cx == 0) near |= 0x49u;
                if (cx == nx - 1) near |= 0x124u;
                if (x == 0) d |= kInletBit;
            }
            cell[m] = d | near;
        }
        float rho, ux, uy;
        phys_moments<FORCE, SC>(a, g, rho, ux, uy);
        phys_collide<FORCE, SC>(a, g, rho, ux, uy);
#pragma unroll
        for (int i = 0; i < 9; ++i) lds[i][r * RW + q] = Dom<T, SC>::out(g[i], a.scale);
    }
    __syncthreads();

    // One step of the region cell c from LDS into gm.
    auto collide = [&](float* gm) {
        float rho, ux, uy;
        phys_moments<FORCE, SC>(a, gm, rho, ux, uy);
        phys_collide<FORCE, SC>(a, gm, rho, ux, uy);
    };
    auto step_lds = [&](int c, uint32_t d, float* gm) {
        // a wavefront without a special cell takes the plain gather
        if (!__any((d & kSlowMask) != 0u)) {
#pragma unroll
            for (int i = 0; i < 9; ++i) gm[i] = Dom<T, SC>::in(lds[i][c - ey_of(i) * RW - ex_of(i)], a.inv_scale);
            // a copy of the collision here lets its first operations take the
            // binary16 values as they come; joined with the other branch each
            // is converted, and packed and unpacked, first
            if constexpr (SC) {
                collide(gm);
                return;
            }
        } else {
            const int cc = (XEDGE == 1 && (d & kOutletBit)) ? c - 1 : c;
            gm[0] = Dom<T, SC>::in(lds[0][cc], a.inv_scale);
#pragma unroll
            for (int i = 1; i < 9; ++i)
                gm[i] = Dom<T, SC>::in(pick(d, pull_bit(i), lds[inv_of(i)][cc], lds[i][cc - ey_of(i) * RW - ex_of(i)]),
                                       a.inv_scale);
            if (XEDGE == 1 && (d & kInletBit)) zou_he_inlet<SC>(a, gm);
        }
        collide(gm);
    };

#pragma unroll
    for (int s = 1; s < RING; ++s) {  // steps 2 .. NS - 1: cells s in from the rim
        const bool qin = q >= s && q < RW - s;
        T out[CPT][9];
#pragma unroll
        for (int m = 0; m < CPT; ++m) {
            const int r = rq + RSTEP * m;
            if (r >= s && r < RH - s && qin && (cell[m] & kLiveBit)) {
                float g[9];
                step_lds(r * RW + q, cell[m], g);
#pragma unroll
                for (int i = 0; i < 9; ++i) out[m][i] = Dom<T, SC>::out(g[i], a.scale);
            }
        }
        __syncthreads();
#pragma unroll
        for (int m = 0; m < CPT; ++m) {
            const int r = rq + RSTEP * m;
            if (r >= s && r < RH - s && qin && (cell[m] & kLiveBit)) {
#pragma unroll
                for (int i = 0; i < 9; ++i) lds[i][r * RW + q] = out[m][i];
            }
        }
        __syncthreads();
    }

    // Step NS: the tile, stored to HBM with the pushes.
    if (q < RING || q >= RW - RING || xr >= nx) return;
#pragma unroll
    for (int m = 0; m < CPT; ++m) {
        const int r = rq + RSTEP * m;
        const int y = y0 - RING + r;
        if (r < RING || r >= RH - RING || y >= ny || !(cell[m] & kLiveBit)) continue;
        float g[9];
        step_lds(r * RW + q, cell[m], g);
        const uint32_t row = __umul24((uint32_t)y, a.rs);
#pragma unroll
        for (int i = 0; i < 9; ++i)
            st<(FLAGS & kNtStore) != 0>(elem<kRowWave>(dst, row, xr, (ptrdiff_t)((uint32_t)i * a.plane)),
                                        Dom<T, SC>::out(g[i], a.scale));
        const uint32_t near = cell[m] >> kNearShift;
        if (near & 0x1EFu) {
            CellNbr nb;
            nb.ym = (y == 0) ? ny - 1 : y - 1;
            nb.yp = (y == ny - 1) ? 0 : y + 1;
            nb.sm = near & 7u;
            nb.s0 = (near >> 3) & 7u;
            nb.sp = (near >> 6) & 7u;
            cell_push<T, XEDGE, SC>(a, dst, nb, xr, y, g);
        }
    }
}

template <typename T, int XEDGE, bool FORCE, int BS, int RW, int RH, int NS, int FLAGS>
// eight waves per SIMD (64 registers), or the one block per CU that fits
__global__ __launch_bounds__(BS, 9 * RW * RH * sizeof(T) > 81920 ? 4 : 8) void k_phys_stepn(PhysArgs a, const T* __restrict__ src, T* __restrict__ dst,
                                                      const uint32_t* __restrict__ bits, uint32_t words,
                                                      uint32_t tiles_x)
{
    __shared__ T lds[9][RW * RH];
    const uint32_t t = (FLAGS & kXcdRemap) ? xcd_remap(blockIdx.x, gridDim.x) : blockIdx.x;
    const int x0 = (int)(t % tiles_x) * (RW - 2 * (NS - 1));
    const int y0 = (int)(t / tiles_x) * (RH - 2 * (NS - 1));
    nstep_tile<T, XEDGE, FORCE, BS, RW, RH, NS, FLAGS>(a, src, dst, bits, words, x0, y0, lds);
}

template <typename T, int XEDGE, bool FORCE, int BS, int RW, int RH, int NS, int FLAGS>
static hipError_t launch_phys_variantn(const PhysArgs& a, const void* src, void* dst, const uint32_t* bits,
                                       uint32_t words, hipStream_t s)
{
    constexpr int BW = RW - 2 * (NS - 1), BH = RH - 2 * (NS - 1);
    if (!nstep_fits(BW, NS, a.nx, a.ny, XEDGE)) return hipErrorInvalidValue;
    const uint32_t tiles_x = (uint32_t)((a.nx + BW - 1) / BW);
    const uint32_t tiles = tiles_x * (uint32_t)((a.ny + BH - 1) / BH);
    hipLaunchKernelGGL((k_phys_stepn<T, XEDGE, FORCE, BS, RW, RH, NS, FLAGS>), dim3(tiles), dim3(BS), 0, s, a,
                       (const T*)src, (T*)dst, bits, words, tiles_x);
    return hipGetLastError();
}

template <typename T, int XEDGE, bool FORCE>
static hipError_t dispatch_variantn(int v, const PhysArgs& a, const void* src, void* dst, const uint32_t* bits,
                                    uint32_t words, hipStream_t s)
{
    constexpr int R = kXcdRemap;
    switch (v) {
    case 48: return launch_phys_variantn<T, XEDGE, FORCE, 1024, 32, 32, 9, 0>(a, src, dst, bits, words, s);
    case 49: return launch_phys_variantn<T, XEDGE, FORCE, 1024, 32, 32, 5, R>(a, src, dst, bits, words, s);
    case 50: return launch_phys_variantn<T, XEDGE, FORCE, 1024, 64, 32, 5, R>(a, src, dst, bits, words, s);
    case 51: return launch_phys_variantn<T, XEDGE, FORCE, 1024, 64, 48, 5, R>(a, src, dst, bits, words, s);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_phys_stepn(int variant, bool f16, int xedge, bool force, const PhysArgs& a, const void* src,
                             void* dst, const uint32_t* bits, uint32_t words, hipStream_t s)
{
#define LBM_DN(T, XE, FO) return dispatch_variantn<T, XE, FO>(variant, a, src, dst, bits, words, s)
    if (f16) {
        if (xedge) { if (force) LBM_DN(_Float16, 1, true); else LBM_DN(_Float16, 1, false); }
        else { if (force) LBM_DN(_Float16, 0, true); else LBM_DN(_Float16, 0, false); }
    }
    if (xedge) { if (force) LBM_DN(float, 1, true); else LBM_DN(float, 1, false); }
    if (force) LBM_DN(float, 0, true);
    LBM_DN(float, 0, false);
#undef LBM_DN
}

// ---------------------------------------------------------------------------
// Batched domains: one block per tile of one domain (tile_dom[t]; domain d
// owns tiles [tile0, tile0 + ceil(nx/BW) ceil(ny/BH))), each domain with its
// own size, tau, inlet, force and x edge.  Microseconds per step of 20 uneven
// channels of 64 to 1024 cells a side (6.1 million cells), the fastest
// three-step shape before, then 31, 32, 33: binary32 38.8, 29.1, 25.1, 34.5;
// binary16 30.8, 27.9, 25.4, 25.1; of 6 channels up to 320: 3.80, 2.23, 2.68,
// 3.57.
// ---------------------------------------------------------------------------
template <typename T, int BS, int RW, int RH, int NS, int FLAGS>
__global__ __launch_bounds__(BS, 9 * RW * RH * sizeof(T) > 81920 ? 4 : 8) void k_batch_stepn(
    const BatchDomainDev* __restrict__ doms, const uint16_t* __restrict__ tile_dom, const T* __restrict__ src,
    T* __restrict__ dst, const uint32_t* __restrict__ bits)
{
    __shared__ T lds[9][RW * RH];
    constexpr int BW = RW - 2 * (NS - 1), BH = RH - 2 * (NS - 1);
    const uint32_t t = (FLAGS & kXcdRemap) ? xcd_remap(blockIdx.x, gridDim.x) : blockIdx.x;
    const BatchDomainDev& D = doms[tile_dom[t]];
    const uint32_t local = t - D.tile0;
    const uint32_t tiles_x = ((uint32_t)D.a.nx + (uint32_t)(BW - 1)) / (uint32_t)BW;
    const int x0 = (int)(local % tiles_x) * BW, y0 = (int)(local / tiles_x) * BH;
    const T* const s = src + D.pop_off;
    T* const o = dst + D.pop_off;
    const uint32_t* const m = bits + D.bits_off;
    if (D.x_edge) {
        if (D.force) nstep_tile<T, 1, true, BS, RW, RH, NS, FLAGS>(D.a, s, o, m, D.words, x0, y0, lds);
        else nstep_tile<T, 1, false, BS, RW, RH, NS, FLAGS>(D.a, s, o, m, D.words, x0, y0, lds);
    } else {
        if (D.force) nstep_tile<T, 0, true, BS, RW, RH, NS, FLAGS>(D.a, s, o, m, D.words, x0, y0, lds);
        else nstep_tile<T, 0, false, BS, RW, RH, NS, FLAGS>(D.a, s, o, m, D.words, x0, y0, lds);
    }
}

template <typename T>
static hipError_t launch_batchn_typed(int v, const BatchDomainDev* doms, const uint16_t* tile_dom, uint32_t ntiles,
                                      const void* src, void* dst, const uint32_t* bits, hipStream_t s)
{
    if (ntiles == 0) return hipSuccess;
#define LBM_BATCHN(BS, RW, RH, NS, FL)                                                                          \
    hipLaunchKernelGGL((k_batch_stepn<T, BS, RW, RH, NS, FL>), dim3(ntiles), dim3(BS), 0, s, doms, tile_dom,    \
                       (const T*)src, (T*)dst, bits)
    switch (v) {
    case 31: LBM_BATCHN(1024, 32, 32, 5, kXcdRemap); break;
    case 32: LBM_BATCHN(1024, 64, 32, 5, kXcdRemap); break;
    case 33: LBM_BATCHN(1024, 64, 48, 5, kXcdRemap); break;
    default: return hipErrorInvalidValue;
    }
#undef LBM_BATCHN
    return hipGetLastError();
}

hipError_t launch_batch_stepn(int variant, bool f16, const BatchDomainDev* doms, const uint16_t* tile_dom,
                              uint32_t ntiles, const void* src, void* dst, const uint32_t* bits, hipStream_t s)
{
    return f16 ? launch_batchn_typed<_Float16>(variant, doms, tile_dom, ntiles, src, dst, bits, s)
               : launch_batchn_typed<float>(variant, doms, tile_dom, ntiles, src, dst, bits, s);
}

}  // namespace lbm
