// lbm_mlp.hip -- the learned collision correction's network: forward,
// backward and Adam kernels (binary32), the sample store, and its C ABI.
//
// No reference counterpart: jinleili/simuverse has no learned collision.
// The network is 9 -> 64 -> 64 -> 9 with GELU (erf form) after both hidden
// layers.  Parameters are one flat vector of 5385 floats:
//     W1[64][9] b1[64] W2[64][64] b2[64] W3[9][64] b3[9]   (row = output)
// The loss of a batch of B samples is L = 1/(9B) sum (y - t)^2.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "lbm.h"
#include "lbm_internal.hpp"

using namespace lbm;

#define MLP_TRY(expr)                                                                               \
    do {                                                                                            \
        hipError_t e_ = (expr);                                                                     \
        if (e_ != hipSuccess) return lbm_fail(LBM_ERR_HIP, "%s: %s", #expr, hipGetErrorString(e_)); \
    } while (0)

namespace lbm {

// SplitMix64 finaliser: sample indices of a minibatch.
__device__ inline uint64_t mix64(uint64_t z)
{
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// ---------------------------------------------------------------------------
// Forward pass (binary32), one sample per thread, weights in LDS.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_mlp_forward(const float* __restrict__ params, const float* __restrict__ X,
                                                     float* __restrict__ Y, int n)
{
    __shared__ float P[kMlpParams];
    for (int k = threadIdx.x; k < kMlpParams; k += 256) P[k] = params[k];
    __syncthreads();
    const int s = blockIdx.x * 256 + threadIdx.x;
    if (s >= n) return;
    float x[kMlpIn], y[kMlpOut];
#pragma unroll
    for (int i = 0; i < kMlpIn; ++i) x[i] = X[(size_t)s * kMlpIn + i];
    mlp_forward_one(P, x, y);
#pragma unroll
    for (int m = 0; m < kMlpOut; ++m) Y[(size_t)s * kMlpOut + m] = y[m];
}

// ---------------------------------------------------------------------------
// Matrix-core forward (bf16 or binary16 operands, binary32 accumulation):
// lane-ordered weights in both operand types are rebuilt from the binary32
// parameters whenever those change; a block of 4 wavefronts takes 256
// samples.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_mlp_pack(const float* __restrict__ params, __bf16* __restrict__ packed,
                                                  _Float16* __restrict__ packed16)
{
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e >= kPackElems) return;
    const float w = pack_weight(params, e);
    packed[e] = (__bf16)w;
    packed16[e] = (_Float16)w;
}

// Stages the packed weights and the biases b1, b2, b3 of a network in LDS.
template <typename E>
__device__ inline void stage_net(const E* __restrict__ packed, const float* __restrict__ params, E* W, float* bias)
{
    const uint4* src = reinterpret_cast<const uint4*>(packed);
    uint4* dst = reinterpret_cast<uint4*>(W);
    for (int k = threadIdx.x; k < kPackElems / 8; k += blockDim.x) dst[k] = src[k];
    for (int k = threadIdx.x; k < kMlpH; k += blockDim.x) {
        bias[k] = params[kOffB1 + k];
        bias[kMlpH + k] = params[kOffB2 + k];
    }
    for (int k = threadIdx.x; k < kBiasElems - 2 * kMlpH; k += blockDim.x)
        bias[2 * kMlpH + k] = k < kMlpOut ? params[kOffB3 + k] : 0.0f;
}

template <typename E>
__global__ __launch_bounds__(256) void k_mlp_forward_mma(const E* __restrict__ packed,
                                                         const float* __restrict__ params,
                                                         const float* __restrict__ X, float* __restrict__ Y, int n)
{
    __shared__ __align__(16) E W[kPackElems];
    __shared__ __align__(16) float bias[kBiasElems];
    __shared__ __align__(16) E xs[4][64 * 16];
    __shared__ float ys[4][64 * kMlpOut];
    stage_net(packed, params, W, bias);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int s = blockIdx.x * 256 + threadIdx.x;
#pragma unroll
    for (int i = 0; i < 16; ++i)
        xs[wave][lane * 16 + i] = (E)((s < n && i < kMlpIn) ? X[(size_t)s * kMlpIn + i] : 0.0f);
    __syncthreads();
    mlp_wave(W, bias, xs[wave], ys[wave], lane);
    __syncthreads();
    if (s >= n) return;
#pragma unroll
    for (int m = 0; m < kMlpOut; ++m) Y[(size_t)s * kMlpOut + m] = ys[wave][lane * kMlpOut + m];
}

// ---------------------------------------------------------------------------
// Loss gradient on matrix cores, binary32 throughout
// (v_mfma_f32_32x32x2_f32 and its 4x4x1 and 16x16x4 forms: binary32
// operands, products and sums).
//
// A wavefront takes 32 samples at a time through the transposed problem
// (rows = units, columns = samples).  Operand layouts, lane l, h = l / 32:
//   32x32x2   A row l % 32, k = h;  B column l % 32, k = h;
//             C value j: column l % 32, row c_row(j, h)
//   16x16x4   A row l % 16, k = l / 16;  B column l % 16, k = l / 16;
//             C value r: column l % 16, row 4 (l / 16) + r
//   4x4x1     16 blocks: A row l % 4, B column l % 4 of block l / 4;
//             C value r: row r, column l % 4 of block l / 4
// C value j of a layer is therefore the next layer's B operand for the K
// pair (c_row(j, 0), c_row(j, 1)), with the weights laid out to match, and
// the forward pass, W3^T dy and W2^T D2 chain in registers.  The weight
// gradients contract over the samples, so their operands need units across
// lanes: each 32 x 32 tile is turned once through a 32 x 36 buffer of the
// wavefront's own (16-byte reads of rows 36 floats apart: no bank
// conflicts), the samples of a K step chosen so that a lane reads four in
// a row.  Layer 1 carries its bias as a tenth input of one, which fills its
// fifth K pair and gives the bias gradient with the weights'.  The nine
// outputs use the 4x4x1 form: block l / 4 holds four samples, the two lane
// halves sum different units and are added at the end.
//
// What bounds it: 16 384 matrix-core cycles per 32 samples and SIMD, 54 % of
// the launch, and the chain around them: the vector instructions (64 GELU and
// derivative pairs per lane) issue for 12 to 14 % and the LDS is busy for 13 %,
// but two wavefronts per SIMD overlap the phases only in part and wait for a
// third of their time.  Each wavefront keeps its sums of the gradient (105
// registers) across its chunks, so memory sees each sample once and one partial
// per block.  All 256 registers are used and 27 values go through scratch
// memory, most of them stored once before the loop over chunks; every store of
// one runs with all lanes on.  Measured on 10^6 samples: 0.40 ms (75 TFLOP/s of
// the 154 a large binary32 matrix product reaches), against 2.25 ms for the
// same sums on the vector ALUs with activations staged in LDS; 4096 samples: 25
// us against 40 us.  Gradient error against binary64 at 4096 samples 3.5e-8
// (1.2e-7 before: the partials of at most 256 blocks are now added in
// binary64); for single samples 2.6e-7 (2.8e-7).
// ---------------------------------------------------------------------------
constexpr int kTS = 32;             // samples a wavefront takes at a time
constexpr int kGradWaves = 8;       // wavefronts per block (two per SIMD)
constexpr int kGradThreads = 64 * kGradWaves;
constexpr int kGradBlocks = 256;    // at most one block per CU
constexpr int kTPad = kTS + 4;      // row stride of the turning buffers
constexpr int kWPad = kMlpH + 4;    // row stride of W2 and W3
// LDS, in floats
constexpr int kLW2 = 0;                         // W2 rows
constexpr int kLW1 = kLW2 + kMlpH * kWPad;      // [W1 | b1] as A: [mt][step][lane]
constexpr int kLW3b = kLW1 + 2 * 5 * 64;        // W3^T as A: [mt][step][lane]
constexpr int kLW3f = kLW3b + 2 * 5 * 64;       // W3 rows, zero-padded to 12
constexpr int kLB2 = kLW3f + 12 * kWPad;
constexpr int kLB3 = kLB2 + kMlpH;              // padded to 12
constexpr int kLWave = kLB3 + 12;               // per wavefront: H1, a turning tile, dy and later x
constexpr int kWaveFloats = (kMlpH + kTS + 10) * kTPad;
constexpr int kGradLds = kLWave + kGradWaves * kWaveFloats;  // 145 KiB
static_assert(kLWave % 4 == 0 && kWaveFloats % 4 == 0, "16-byte aligned buffers");
static_assert(kGradWaves * kWaveFloats >= kMlpParams, "the block's sum reuses the wavefronts' buffers");
static_assert(kGradLds * sizeof(float) + kGradWaves * sizeof(double) <= 160 * 1024, "LDS of one CU");

typedef float f32x4 __attribute__((ext_vector_type(4)));

// Blocks of the gradient of `batch` samples: one 32-sample chunk per
// wavefront until every CU has a block, then chunks in turn (chunk c goes to
// wavefront (c / blocks) % 8 of block c % blocks), so a small batch spreads
// over the CUs and a large one leaves 256 partials.
inline int mlp_grad_blocks(int batch) { return std::min((batch + kTS - 1) / kTS, kGradBlocks); }

// GELU x Phi(x) and its derivative Phi(x) + x phi(x) of one activation from
// one exponential: with e = exp(-x^2/2) and t = 1 / (1 + 0.45 |x|),
//   1 - Phi(|x|) = e (c1 t + c2 t^2 + .. + c7 t^7)
// (the form of Abramowitz & Stegun 7.1.26; coefficients fitted to
// erfcx(|x| / sqrt 2) / 2 by reweighted least squares, largest deviation of
// Phi 8.3e-9 before rounding, at |x| = 0.38).  On the device over [-9, 9]
// against binary64: GELU rms 5.6e-8 (largest 3.7e-7, at |x| near 9), derivative
// rms 2.6e-8, as the erff form (6.4e-8, 4.5e-7, 2.4e-8).  No branch: 17 vector
// instructions, where erff and expf take about 80 with both sides of erff's
// branch.
__device__ __forceinline__ void gelu_both(float x, float& y, float& d)
{
    const float t = __builtin_amdgcn_rcpf(fmaf(fabsf(x), 0.45f, 1.0f));
    float p = -0.03785362467169762f;
    p = fmaf(p, t, 0.21744582056999207f);
    p = fmaf(p, t, -0.47403931617736816f);
    p = fmaf(p, t, 0.39363744854927063f);
    p = fmaf(p, t, 0.01813739538192749f);
    p = fmaf(p, t, 0.20540063083171844f);
    p = fmaf(p, t, 0.17727164924144745f);
    const float e = __builtin_amdgcn_exp2f((x * x) * -0.72134752044448170f);
    const float q = (p * t) * e;
    const float phi = x >= 0.0f ? 1.0f - q : q;
    y = x * phi;
    d = fmaf(x * e, 0.39894228040143268f, phi);
}

// Orders a wavefront's LDS writes before its lanes' reads of one another's
// (the LDS executes one wavefront's accesses in order; this only keeps the
// compiler from moving them).
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Turns one C tile (rows = units) into rows of the wavefront's buffer.
__device__ __forceinline__ void put_tile(float* __restrict__ tb, const f32x16& c, int lane)
{
    const int h = lane >> 5, n = lane & 31;
    wave_lds_fence();  // earlier reads of the buffer
#pragma unroll
    for (int j = 0; j < 16; ++j) tb[c_row(j, h) * kTPad + n] = c[j];
    wave_lds_fence();
}

__global__ __launch_bounds__(kGradThreads, 2) void k_mlp_grad_partial(
    const float* __restrict__ params, const float* __restrict__ X, const float* __restrict__ T, int n, int batch,
    uint64_t seed, int use_index, float* __restrict__ partial, double* __restrict__ loss_part)
{
    __shared__ __align__(16) float lds[kGradLds];
    __shared__ double lsum[kGradWaves];
    const int tid = (int)threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int h = lane >> 5, c32 = lane & 31, c16 = lane & 15, q16 = lane >> 4;
    // weights in operand order
    for (int e = tid; e < kMlpH * kMlpH; e += kGradThreads)
        lds[kLW2 + (e / kMlpH) * kWPad + e % kMlpH] = params[kOffW2 + e];
    for (int e = tid; e < 2 * 5 * 64; e += kGradThreads) {
        const int l = e & 63, st = (e >> 6) % 5, mt = (e >> 6) / 5;
        const int unit = 32 * mt + (l & 31), k = 2 * st + (l >> 5);
        lds[kLW1 + e] = k < kMlpIn ? params[kOffW1 + unit * kMlpIn + k] : params[kOffB1 + unit];
        lds[kLW3b + e] = k < kMlpOut ? params[kOffW3 + k * kMlpH + unit] : 0.0f;
    }
    for (int e = tid; e < 12 * kWPad; e += kGradThreads) {
        const int m = e / kWPad, k = e % kWPad;
        lds[kLW3f + e] = m < kMlpOut && k < kMlpH ? params[kOffW3 + m * kMlpH + k] : 0.0f;
    }
    if (tid < kMlpH) lds[kLB2 + tid] = params[kOffB2 + tid];
    if (tid < 12) lds[kLB3 + tid] = tid < kMlpOut ? params[kOffB3 + tid] : 0.0f;
    float* const hb = lds + kLWave + wave * kWaveFloats;
    float* const tb = hb + kMlpH * kTPad;
    float* const sb = tb + kTS * kTPad;
    // row of a 10-row operand in the 16-row forms: the results of rows 10..15 are not used
    const int r10 = min(c16, 9);
    __syncthreads();

    f32x16 aW2[2][2];
    f32x4 aW1[4], aW3[4];
    float aB2[2] = {0.0f, 0.0f}, aB3[5] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    double lacc = 0.0;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) aW2[i][j][e] = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) aW1[i] = aW3[i] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};

    const float inv = 2.0f / (9.0f * (float)batch);
    const int nchunks = (batch + kTS - 1) / kTS;
    const int grid = (int)gridDim.x;
    for (int chunk = wave * grid + (int)blockIdx.x; chunk < nchunks; chunk += kGradWaves * grid) {
        const int g = chunk * kTS + c32;  // position in the batch
        const bool live = g < batch;
        // sample index: the batch position itself, or a hashed draw from n
        const int idx = !live ? 0
                              : (use_index ? (int)(mix64(seed + 0x9E3779B97F4A7C15ull * (uint64_t)(g + 1)) % (uint64_t)n)
                                           : g);
        // inputs 2 s + h (the tenth is one)
        float x[5];
#pragma unroll
        for (int s = 0; s < 5; ++s) {
            const int k = 2 * s + h;
            const float v = X[(size_t)idx * kMlpIn + min(k, kMlpIn - 1)];
            x[s] = k == kMlpIn ? 1.0f : (live ? v : 0.0f);
        }

        // layer 1: H1 and GELU'
        f32x16 h1[2], d1[2];
#pragma unroll
        for (int mt = 0; mt < 2; ++mt) {
            f32x16 c;
#pragma unroll
            for (int j = 0; j < 16; ++j) c[j] = 0.0f;
#pragma unroll
            for (int s = 0; s < 5; ++s)
                c = __builtin_amdgcn_mfma_f32_32x32x2f32(lds[kLW1 + (mt * 5 + s) * 64 + lane], x[s], c, 0, 0, 0);
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                float y, d;
                gelu_both(c[j], y, d);
                h1[mt][j] = y;
                d1[mt][j] = d;
            }
        }
        // layer 2
        f32x16 h2[2], d2[2];
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
            for (int gq = 0; gq < 4; ++gq) {
                const f32x4 v = *reinterpret_cast<const f32x4*>(lds + kLB2 + 32 * mt + 8 * gq + 4 * h);
#pragma unroll
                for (int e = 0; e < 4; ++e) h2[mt][4 * gq + e] = v[e];
            }
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int gq = 0; gq < 4; ++gq) {
                f32x4 w[2];
#pragma unroll
                for (int mt = 0; mt < 2; ++mt)
                    w[mt] = *reinterpret_cast<const f32x4*>(lds + kLW2 + (32 * mt + c32) * kWPad + 32 * kt + 8 * gq +
                                                            4 * h);
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int mt = 0; mt < 2; ++mt)
                        h2[mt] = __builtin_amdgcn_mfma_f32_32x32x2f32(w[mt][e], h1[kt][4 * gq + e], h2[mt], 0, 0, 0);
            }
        // H1 for W2's gradient
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) put_tile(hb + 32 * kt * kTPad, h1[kt], lane);
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                float y, d;
                gelu_both(h2[mt][j], y, d);
                h2[mt][j] = y;
                d2[mt][j] = d;
            }
        // outputs: value r of y[o] is output 4 o + r of sample c32, over the
        // units of lane half h
        f32x4 y[3];
#pragma unroll
        for (int o = 0; o < 3; ++o)
#pragma unroll
            for (int r = 0; r < 4; ++r) y[o][r] = h == 0 ? lds[kLB3 + 4 * o + r] : 0.0f;
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int gq = 0; gq < 4; ++gq) {
                f32x4 w[3];
#pragma unroll
                for (int o = 0; o < 3; ++o)
                    w[o] = *reinterpret_cast<const f32x4*>(lds + kLW3f + (4 * o + (lane & 3)) * kWPad + 32 * kt + 8 * gq +
                                                           4 * h);
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int o = 0; o < 3; ++o)
                        y[o] = __builtin_amdgcn_mfma_f32_4x4x1f32(w[o][e], h2[kt][4 * gq + e], y[o], 0, 0, 0);
            }
        // residual of output 2 s + h, and dL/dy
        float dy[5];
#pragma unroll
        for (int s = 0; s < 5; ++s) {
            // the two halves' sums of outputs 2 s and 2 s + 1
            const float a = y[(2 * s) >> 2][(2 * s) & 3], b = y[(2 * s + 1) >> 2][(2 * s + 1) & 3];
            const float own = h == 0 ? a : b, other = h == 0 ? b : a;
            const float v = own + __shfl_xor(other, 32, 64);
            const float t = T[(size_t)idx * kMlpOut + min(2 * s + h, kMlpOut - 1)];
            const float r = live && 2 * s + h < kMlpOut ? v - t : 0.0f;
            lacc += (double)r * (double)r;
            dy[s] = r * inv;
            aB3[s] += dy[s];
        }
        wave_lds_fence();
#pragma unroll
        for (int s = 0; s < 5; ++s) sb[(2 * s + h) * kTPad + c32] = dy[s];
        wave_lds_fence();
        // W3's gradient: dy H2^T, sample 8 (l / 16) + i in K step i
        {
            float dyt[8];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const f32x4 v = *reinterpret_cast<const f32x4*>(sb + r10 * kTPad + 8 * q16 + 4 * i);
#pragma unroll
                for (int e = 0; e < 4; ++e) dyt[4 * i + e] = v[e];
            }
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) {
                put_tile(tb, h2[kt], lane);
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        const f32x4 v = *reinterpret_cast<const f32x4*>(tb + (16 * u + c16) * kTPad + 8 * q16 + 4 * i);
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            aW3[2 * kt + u] =
                                __builtin_amdgcn_mfma_f32_16x16x4f32(dyt[4 * i + e], v[e], aW3[2 * kt + u], 0, 0, 0);
                    }
            }
        }
        // D2 = (W3^T dy) GELU'(A2)
#pragma unroll
        for (int mt = 0; mt < 2; ++mt) {
            f32x16 c;
#pragma unroll
            for (int j = 0; j < 16; ++j) c[j] = 0.0f;
#pragma unroll
            for (int s = 0; s < 5; ++s)
                c = __builtin_amdgcn_mfma_f32_32x32x2f32(lds[kLW3b + (mt * 5 + s) * 64 + lane], dy[s], c, 0, 0, 0);
#pragma unroll
            for (int j = 0; j < 16; ++j) d2[mt][j] *= c[j];
        }
        // W2's gradient: D2 H1^T, sample 16 h + i in K step i
#pragma unroll
        for (int mt = 0; mt < 2; ++mt) {
            put_tile(tb, d2[mt], lane);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const f32x4 v = *reinterpret_cast<const f32x4*>(tb + c32 * kTPad + 16 * h + 4 * i);
                f32x4 u[2];
#pragma unroll
                for (int nt = 0; nt < 2; ++nt)
                    u[nt] = *reinterpret_cast<const f32x4*>(hb + (32 * nt + c32) * kTPad + 16 * h + 4 * i);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    aB2[mt] += v[e];
#pragma unroll
                    for (int nt = 0; nt < 2; ++nt)
                        aW2[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x2f32(v[e], u[nt][e], aW2[mt][nt], 0, 0, 0);
                }
            }
        }
        // D1 = (W2^T D2) GELU'(A1)
        f32x16 cc[2];
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
            for (int j = 0; j < 16; ++j) cc[mt][j] = 0.0f;
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int j = 0; j < 16; ++j) {
#pragma unroll
                for (int mt = 0; mt < 2; ++mt)
                    cc[mt] = __builtin_amdgcn_mfma_f32_32x32x2f32(
                        lds[kLW2 + (32 * kt + c_row(j, h)) * kWPad + 32 * mt + c32], d2[kt][j], cc[mt], 0, 0, 0);
            }
        // [W1 | b1]'s gradient: D1 [x 1]^T, sample 8 (l / 16) + i in K step i
        wave_lds_fence();
#pragma unroll
        for (int s = 0; s < 5; ++s) sb[(2 * s + h) * kTPad + c32] = x[s];
        wave_lds_fence();
        float xt[8];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(sb + r10 * kTPad + 8 * q16 + 4 * i);
#pragma unroll
            for (int e = 0; e < 4; ++e) xt[4 * i + e] = v[e];
        }
#pragma unroll
        for (int mt = 0; mt < 2; ++mt) {
#pragma unroll
            for (int j = 0; j < 16; ++j) cc[mt][j] *= d1[mt][j];
            put_tile(tb, cc[mt], lane);
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const f32x4 v = *reinterpret_cast<const f32x4*>(tb + (16 * u + c16) * kTPad + 8 * q16 + 4 * i);
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        aW1[2 * mt + u] =
                            __builtin_amdgcn_mfma_f32_16x16x4f32(v[e], xt[4 * i + e], aW1[2 * mt + u], 0, 0, 0);
                }
        }
    }

    // The block's sum, wavefront after wavefront over the buffers they no
    // longer need; every parameter has one lane in each wavefront.
    const double ls = wave_sum(lacc);
    if (lane == 0) lsum[wave] = ls;
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) aB2[mt] += __shfl_xor(aB2[mt], 32, 64);
#pragma unroll
    for (int s = 0; s < 5; ++s)
#pragma unroll
        for (int off = 16; off > 0; off >>= 1) aB3[s] += __shfl_xor(aB3[s], off, 64);
    float* const red = lds + kLWave;
    // wavefronts of this block that had a chunk
    const int left = nchunks - (int)blockIdx.x;
    const int active = std::min(kGradWaves, (left + grid - 1) / grid);
    __syncthreads();
    for (int p = tid; p < kMlpParams; p += kGradThreads) red[p] = 0.0f;
    __syncthreads();
    for (int w = 0; w < active; ++w) {
        if (wave == w) {
            auto add = [&](int p, float v) { red[p] += v; };
#pragma unroll
            for (int mt = 0; mt < 2; ++mt) {
#pragma unroll
                for (int nt = 0; nt < 2; ++nt)
#pragma unroll
                    for (int j = 0; j < 16; ++j)
                        add(kOffW2 + (32 * mt + c_row(j, h)) * kMlpH + 32 * nt + c32, aW2[mt][nt][j]);
                if (h == 0) add(kOffB2 + 32 * mt + c32, aB2[mt]);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int unit = 16 * i + 4 * q16 + r;
                    if (c16 < kMlpIn) add(kOffW1 + unit * kMlpIn + c16, aW1[i][r]);
                    else if (c16 == kMlpIn) add(kOffB1 + unit, aW1[i][r]);
                    const int m = 4 * q16 + r;
                    if (m < kMlpOut) add(kOffW3 + m * kMlpH + 16 * i + c16, aW3[i][r]);
                }
#pragma unroll
            for (int s = 0; s < 5; ++s)
                if (c32 == 0 && 2 * s + h < kMlpOut) add(kOffB3 + 2 * s + h, aB3[s]);
        }
        __syncthreads();
    }
    float* out = partial + (size_t)blockIdx.x * kMlpParams;
    for (int p = tid; p < kMlpParams; p += kGradThreads) out[p] = red[p];
    if (tid == 0) {
        double l = 0.0;
        for (int w = 0; w < kGradWaves; ++w) l += lsum[w];
        loss_part[blockIdx.x] = l;
    }
}

// grad[p] = sum over blocks of partial[b][p], in binary64 and a fixed order:
// 64 parameters per block of 1024 threads, wavefront w adding partials w,
// w + 16, ...  (85 blocks with 16 rows in flight each; one thread per
// parameter walking all of the partials took 0.27 ms for 1024 of them.)
__global__ __launch_bounds__(1024) void k_mlp_grad_reduce(const float* __restrict__ partial, int nblocks,
                                                          float* __restrict__ grad,
                                                          const double* __restrict__ loss_part,
                                                          double* __restrict__ loss, int batch)
{
    __shared__ double sh[16][64];
    const int lane = (int)(threadIdx.x & 63u), w = (int)(threadIdx.x >> 6);
    const int p = (int)blockIdx.x * 64 + lane;
    double acc = 0.0;
    if (p < kMlpParams) {
#pragma unroll 4
        for (int b = w; b < nblocks; b += 16) acc += (double)partial[(size_t)b * kMlpParams + p];
    }
    sh[w][lane] = acc;
    __syncthreads();
    if (w == 0 && p < kMlpParams) {
        double s = 0.0;
#pragma unroll
        for (int k = 0; k < 16; ++k) s += sh[k][lane];
        grad[p] = (float)s;
    }
    if (blockIdx.x == 0 && w == 1) {
        double l = 0.0;
        for (int b = lane; b < nblocks; b += 64) l += loss_part[b];
        l = wave_sum(l);
        if (lane == 0) *loss = l / (9.0 * (double)batch);
    }
}

// Sum of squares of a[0..count) in binary64: grid-stride, one partial per
// block (the host adds the partials in block order).
__global__ __launch_bounds__(256) void k_sumsq(const float* __restrict__ a, size_t count, double* __restrict__ partial)
{
    double acc = 0.0;
    for (size_t k = blockIdx.x * 256ull + threadIdx.x; k < count; k += (size_t)gridDim.x * 256ull)
        acc += (double)a[k] * (double)a[k];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
    __shared__ double sh[4];
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) partial[blockIdx.x] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

__global__ __launch_bounds__(256) void k_scale(float* __restrict__ a, size_t count, float s)
{
    for (size_t k = blockIdx.x * 256ull + threadIdx.x; k < count; k += (size_t)gridDim.x * 256ull) a[k] *= s;
}

// Adam (Kingma & Ba 2015, Algorithm 1) on the binary32 master parameters
// and moments; the arithmetic between them is binary64, so a step rounds
// each of the three once.
__global__ __launch_bounds__(256) void k_mlp_adam(float* __restrict__ p, const float* __restrict__ g,
                                                  float* __restrict__ m, float* __restrict__ v, double lr, double b1,
                                                  double b2, double eps, double c1, double c2)
{
    const int k = blockIdx.x * 256 + threadIdx.x;
    if (k >= kMlpParams) return;
    const double gk = (double)g[k];
    const double mk = b1 * (double)m[k] + (1.0 - b1) * gk;
    const double vk = b2 * (double)v[k] + (1.0 - b2) * gk * gk;
    m[k] = (float)mk;
    v[k] = (float)vk;
    p[k] = (float)((double)p[k] - lr * (mk / c1) / (sqrt(vk / c2) + eps));
}

// ---------------------------------------------------------------------------
// Samples from a pair of coarse pre-collision states (state_t, state_t1,
// dense host layout f[i*n + c], binary32 f):
//   features  x_i = (f_i - feq_i) / (w_i s_in)          at cell c, time t
//   target    t_i = P(f_i(c + e_i, t+1) - BGK_i(f(c, t))) / (w_i s_out)
// where P removes the mass and momentum of a correction.  Cells that are
// solid or have a solid neighbour are skipped; y and x are periodic.
// Candidate k is cell k * stride + offset.  The samples are stored in
// candidate order (a count pass, an exclusive scan of the per-block counts,
// then each block writes at its base in thread order), so the sample set,
// and the training that draws from it, are the same on every run.
// ---------------------------------------------------------------------------
__device__ inline bool transition_cell(const uint8_t* __restrict__ solid, int nx, int ny, uint32_t k,
                                       uint32_t stride, uint32_t offset, uint32_t& c)
{
    const uint32_t n = (uint32_t)nx * (uint32_t)ny;
    const uint64_t c64 = (uint64_t)k * stride + offset;
    if (c64 >= n) return false;
    c = (uint32_t)c64;
    const int y = (int)(c / (uint32_t)nx), x = (int)(c % (uint32_t)nx);
    for (int dy2 = -1; dy2 <= 1; ++dy2)
        for (int dx2 = -1; dx2 <= 1; ++dx2) {
            const int xx = (x + dx2 + nx) % nx, yy = (y + dy2 + ny) % ny;
            if (solid[(uint32_t)yy * nx + xx]) return false;
        }
    return true;
}

__global__ __launch_bounds__(256) void k_mlp_transition_count(const uint8_t* __restrict__ solid, int nx, int ny,
                                                              uint32_t stride, uint32_t offset, int* __restrict__ counts)
{
    uint32_t c = 0;
    const bool take = transition_cell(solid, nx, ny, blockIdx.x * 256u + threadIdx.x, stride, offset, c);
    const int total = __syncthreads_count(take ? 1 : 0);
    if (threadIdx.x == 0) counts[blockIdx.x] = total;
}

// block_base: first slot of each block's samples (the running sample count
// plus the exclusive scan of the counts, clamped to max_samples).
__global__ __launch_bounds__(256) void k_mlp_transition(const float* __restrict__ s0, const float* __restrict__ s1,
                                                        const uint8_t* __restrict__ solid, PhysArgs a, float s_in,
                                                        float s_out, uint32_t stride, uint32_t offset,
                                                        int max_samples, const int* __restrict__ block_base,
                                                        float* __restrict__ X, float* __restrict__ T)
{
    __shared__ int wave_total[4];
    const int nx = a.nx, ny = a.ny;
    const uint32_t n = (uint32_t)nx * (uint32_t)ny;
    uint32_t c = 0;
    const bool take = transition_cell(solid, nx, ny, blockIdx.x * 256u + threadIdx.x, stride, offset, c);
    // rank of this cell among the block's samples, in thread order
    const int lane = (int)(threadIdx.x & 63u), wave = (int)(threadIdx.x >> 6);
    const uint64_t mask = __ballot(take ? 1 : 0);
    const int below = __popcll(mask & ((1ull << lane) - 1ull));
    if (lane == 0) wave_total[wave] = __popcll(mask);
    __syncthreads();
    if (!take) return;
    int rank = below;
    for (int w = 0; w < wave; ++w) rank += wave_total[w];
    const int y = (int)(c / (uint32_t)nx), x = (int)(c % (uint32_t)nx);
    // The step's own arithmetic on deviations g = f - w: moments, features,
    // BGK (+ Guo).
    float g[9], gc[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) g[i] = s0[(size_t)i * n + c] - w_phys(i);
    float rho, ux, uy;
    phys_moments<true>(a, g, rho, ux, uy);
    float xin[9], d[9], nm[3], inv_ws[3];
    learned_input_scales(s_in, inv_ws);
    learned_inputs(g, rho, ux, uy, inv_ws, xin, nm);
#pragma unroll
    for (int i = 0; i < 9; ++i) gc[i] = g[i];
    phys_collide<true>(a, gc, rho, ux, uy);
#pragma unroll
    for (int i = 0; i < 9; ++i) {
        const int tx = (x + ex_of(i) + nx) % nx, ty = (y + ey_of(i) + ny) % ny;
        d[i] = (s1[(size_t)i * n + (uint32_t)ty * nx + tx] - w_phys(i)) - gc[i];
    }
    // Targets of the three modulations (add_stress_correction): residual
    // moment over non-equilibrium moment, d_a / n_a, regularised where n_a
    // is small against the cell's stress: d_a n_a / (n_a^2 + eps^2) with
    // eps^2 = 1e-2 (n_xx^2 + n_xy^2 + n_e^2 / 9), clamped to the bounds the
    // step applies.  nm holds n_e, n_xx, n_xy (learned_inputs).
    float de = 0.0f, dxx = 0.0f, dxy = 0.0f;
#pragma unroll
    for (int i = 0; i < 9; ++i) {
        const float ex = (float)ex_of(i), ey = (float)ey_of(i);
        de += mom_e(i) * d[i];
        dxx += (ex * ex - ey * ey) * d[i];
        dxy += (ex * ey) * d[i];
    }
    const float ne = nm[0], nxx = nm[1], nxy = nm[2];
    const float eps2 = 1e-2f * (nxx * nxx + nxy * nxy + ne * ne * (1.0f / 9.0f)) + 1e-30f;
    const float lo = modulation_lo(a.omega), hi = modulation_hi(a.omega);
    auto ratio = [&](float dm, float n_a) { return fminf(fmaxf(dm * n_a / (n_a * n_a + eps2), lo), hi); };
    float t[9] = {ratio(de, ne), ratio(dxx, nxx), ratio(dxy, nxy), 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    const int slot = block_base[blockIdx.x] + rank;
    if (slot >= max_samples) return;
#pragma unroll
    for (int i = 0; i < 9; ++i) {
        X[(size_t)slot * 9 + i] = xin[i];
        T[(size_t)slot * 9 + i] = t[i] / s_out;
    }
}

}  // namespace lbm

struct lbm_mlp {
    int dev = 0;
    hipStream_t stream = nullptr;
    float* params = nullptr;  // binary32 master copy
    __bf16* packed = nullptr;      // lane-ordered bf16 weights of the matrix-core path
    _Float16* packed16 = nullptr;  // the same in binary16
    float* adam_m = nullptr;
    float* adam_v = nullptr;
    float* grad = nullptr;
    float* partial = nullptr;  // per-block gradient partials
    double* loss_part = nullptr;
    double* loss = nullptr;
    int partial_blocks = 0;
    float* X = nullptr;  // samples
    float* T = nullptr;
    int capacity = 0;
    int samples = 0;
    int adam_step = 0;
    float s_in = 1.0f, s_out = 1.0f;
    // Bumped whenever the parameters or scales change: lattices with this
    // network attached rebuild the HIP graphs they captured (a graph holds
    // the scales its launches were recorded with).
    uint64_t generation = 0;
};

namespace {

int mlp_check(lbm_mlp* m)
{
    if (!m) return lbm_fail(LBM_ERR_INVALID, "null network");
    MLP_TRY(hipSetDevice(m->dev));
    return LBM_OK;
}

// Before the parameters change: lattices on other streams may still be
// running learned steps that read them, so every queue of the device drains
// first.  (Updates are rare next to steps; the wait costs one round trip.)
int mlp_quiesce_device(lbm_mlp* m)
{
    MLP_TRY(hipDeviceSynchronize());
    return LBM_OK;
}

void mlp_free(lbm_mlp* m)
{
    for (void* p : {(void*)m->params, (void*)m->packed, (void*)m->packed16, (void*)m->adam_m, (void*)m->adam_v, (void*)m->grad, (void*)m->partial,
                    (void*)m->loss_part, (void*)m->loss, (void*)m->X, (void*)m->T})
        if (p) (void)hipFree(p);
    if (m->stream) (void)hipStreamDestroy(m->stream);
    delete m;
}

// Gradient of the loss over `batch` samples (the first `batch` stored
// samples, or hashed draws when use_index) into m->grad; loss into m->loss.
int mlp_grad(lbm_mlp* m, const float* X, const float* T, int n, int batch, uint64_t seed, int use_index)
{
    const int nb = mlp_grad_blocks(batch);
    if (nb > m->partial_blocks) {
        if (m->partial) (void)hipFree(m->partial);
        if (m->loss_part) (void)hipFree(m->loss_part);
        m->partial = nullptr;
        m->loss_part = nullptr;
        m->partial_blocks = 0;  // until both are there
        MLP_TRY(hipMalloc(&m->partial, (size_t)nb * kMlpParams * sizeof(float)));
        MLP_TRY(hipMalloc(&m->loss_part, (size_t)nb * sizeof(double)));
        m->partial_blocks = nb;
    }
    hipLaunchKernelGGL(k_mlp_grad_partial, dim3(nb), dim3(kGradThreads), 0, m->stream, m->params, X, T, n, batch, seed,
                       use_index, m->partial, m->loss_part);
    MLP_TRY(hipGetLastError());
    hipLaunchKernelGGL(k_mlp_grad_reduce, dim3((kMlpParams + 63) / 64), dim3(1024), 0, m->stream, m->partial, nb,
                       m->grad, m->loss_part, m->loss, batch);
    MLP_TRY(hipGetLastError());
    return LBM_OK;
}

// Rebuilds the matrix-core weights after the binary32 parameters changed.
int mlp_repack(lbm_mlp* m)
{
    hipLaunchKernelGGL(k_mlp_pack, dim3((kPackElems + 255) / 256), dim3(256), 0, m->stream, m->params, m->packed,
                       m->packed16);
    MLP_TRY(hipGetLastError());
    return LBM_OK;
}

}  // namespace

const __bf16* lbm_mlp_device_packed(const lbm_mlp* m) { return m->packed; }
const _Float16* lbm_mlp_device_packed16(const lbm_mlp* m) { return m->packed16; }

// Device pointer to the binary32 parameters and the two scales of a
// network (used by the learned collision step).
const float* lbm_mlp_device_params(const lbm_mlp* m) { return m->params; }
void lbm_mlp_scales(const lbm_mlp* m, float* s_in, float* s_out)
{
    *s_in = m->s_in;
    *s_out = m->s_out;
}
uint64_t lbm_mlp_generation(const lbm_mlp* m) { return m->generation; }

extern "C" {

int lbm_mlp_param_count(void) { return kMlpParams; }

int lbm_mlp_create(uint64_t seed, int capacity, lbm_mlp** out)
{
    if (!out) return lbm_fail(LBM_ERR_INVALID, "null out");
    *out = nullptr;
    if (capacity < 0) return lbm_fail(LBM_ERR_INVALID, "capacity must be >= 0");
    lbm_mlp* m = new lbm_mlp();
    hipError_t e = hipGetDevice(&m->dev);
    if (e == hipSuccess) e = hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking);
    const size_t pb = kMlpParams * sizeof(float);
    if (e == hipSuccess) e = hipMalloc(&m->params, pb);
    if (e == hipSuccess) e = hipMalloc(&m->packed, kPackElems * sizeof(__bf16));
    if (e == hipSuccess) e = hipMalloc(&m->packed16, kPackElems * sizeof(_Float16));
    if (e == hipSuccess) e = hipMalloc(&m->adam_m, pb);
    if (e == hipSuccess) e = hipMalloc(&m->adam_v, pb);
    if (e == hipSuccess) e = hipMalloc(&m->grad, pb);
    if (e == hipSuccess) e = hipMalloc(&m->loss, sizeof(double));
    if (e == hipSuccess && capacity > 0) e = hipMalloc(&m->X, (size_t)capacity * kMlpIn * sizeof(float));
    if (e == hipSuccess && capacity > 0) e = hipMalloc(&m->T, (size_t)capacity * kMlpOut * sizeof(float));
    if (e != hipSuccess) {
        mlp_free(m);
        return lbm_fail(LBM_ERR_OOM, "network allocation: %s", hipGetErrorString(e));
    }
    m->capacity = capacity;
    // Glorot-uniform weights from SplitMix64(seed), zero biases.
    std::vector<float> p(kMlpParams, 0.0f);
    uint64_t st = seed;
    auto uni = [&]() {
        st += 0x9E3779B97F4A7C15ull;
        uint64_t z = st;
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        z ^= z >> 31;
        return (double)(z >> 11) * (1.0 / 9007199254740992.0);
    };
    auto fill = [&](int off, int fan_out, int fan_in) {
        const double a = std::sqrt(6.0 / (fan_in + fan_out));
        for (int k = 0; k < fan_out * fan_in; ++k) p[off + k] = (float)((2.0 * uni() - 1.0) * a);
    };
    fill(kOffW1, kMlpH, kMlpIn);
    fill(kOffW2, kMlpH, kMlpH);
    fill(kOffW3, kMlpOut, kMlpH);
    e = hipMemcpy(m->params, p.data(), pb, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemset(m->adam_m, 0, pb);
    if (e == hipSuccess) e = hipMemset(m->adam_v, 0, pb);
    if (e != hipSuccess || mlp_repack(m) != LBM_OK || hipStreamSynchronize(m->stream) != hipSuccess) {
        mlp_free(m);
        return lbm_fail(LBM_ERR_HIP, "network init failed");
    }
    *out = m;
    return LBM_OK;
}

int lbm_mlp_destroy(lbm_mlp* m)
{
    if (!m) return LBM_OK;
    (void)hipSetDevice(m->dev);
    if (m->stream) (void)hipStreamSynchronize(m->stream);
    mlp_free(m);
    return LBM_OK;
}

int lbm_mlp_set_params(lbm_mlp* m, const float* params)
{
    int rc = mlp_check(m);
    if (rc) return rc;
    if (!params) return lbm_fail(LBM_ERR_INVALID, "null params");
    if ((rc = mlp_quiesce_device(m))) return rc;
    ++m->generation;
    MLP_TRY(hipMemcpyAsync(m->params, params, kMlpParams * sizeof(float), hipMemcpyHostToDevice, m->stream));
    MLP_TRY(hipMemsetAsync(m->adam_m, 0, kMlpParams * sizeof(float), m->stream));
    MLP_TRY(hipMemsetAsync(m->adam_v, 0, kMlpParams * sizeof(float), m->stream));
    if ((rc = mlp_repack(m))) return rc;
    MLP_TRY(hipStreamSynchronize(m->stream));
    m->adam_step = 0;
    return LBM_OK;
}

int lbm_mlp_get_params(lbm_mlp* m, float* params)
{
    int rc = mlp_check(m);
    if (rc) return rc;
    if (!params) return lbm_fail(LBM_ERR_INVALID, "null params");
    MLP_TRY(hipMemcpyAsync(params, m->params, kMlpParams * sizeof(float), hipMemcpyDeviceToHost, m->stream));
    MLP_TRY(hipStreamSynchronize(m->stream));
    return LBM_OK;
}

int lbm_mlp_set_scales(lbm_mlp* m, float in_scale, float out_scale)
{
    if (!m) return lbm_fail(LBM_ERR_INVALID, "null network");
    if (!(in_scale > 0.0f) || !(out_scale > 0.0f) || !std::isfinite(in_scale) || !std::isfinite(out_scale))
        return lbm_fail(LBM_ERR_INVALID, "scales must be finite and > 0");
    if (in_scale != m->s_in || out_scale != m->s_out) ++m->generation;
    m->s_in = in_scale;
    m->s_out = out_scale;
    return LBM_OK;
}

int lbm_mlp_get_scales(lbm_mlp* m, float* in_scale, float* out_scale)
{
    if (!m || !in_scale || !out_scale) return lbm_fail(LBM_ERR_INVALID, "null argument");
    *in_scale = m->s_in;
    *out_scale = m->s_out;
    return LBM_OK;
}

static int mlp_forward_impl(lbm_mlp* m, const float* x, int n, float* y, int precision)
{
    int rc = mlp_check(m);
    if (rc) return rc;
    if (!x || !y || n < 0) return lbm_fail(LBM_ERR_INVALID, "bad arguments");
    if (n == 0) return LBM_OK;
    float *dx = nullptr, *dy = nullptr;
    MLP_TRY(hipMalloc(&dx, (size_t)n * kMlpIn * sizeof(float)));
    hipError_t e = hipMalloc(&dy, (size_t)n * kMlpOut * sizeof(float));
    if (e == hipSuccess) e = hipMemcpyAsync(dx, x, (size_t)n * kMlpIn * sizeof(float), hipMemcpyHostToDevice, m->stream);
    if (e == hipSuccess) {
        if (precision == LBM_MLP_BF16)
            hipLaunchKernelGGL(k_mlp_forward_mma<__bf16>, dim3((n + 255) / 256), dim3(256), 0, m->stream,
                               m->packed, m->params, dx, dy, n);
        else if (precision == LBM_MLP_F16)
            hipLaunchKernelGGL(k_mlp_forward_mma<_Float16>, dim3((n + 255) / 256), dim3(256), 0, m->stream,
                               m->packed16, m->params, dx, dy, n);
        else
            hipLaunchKernelGGL(k_mlp_forward, dim3((n + 255) / 256), dim3(256), 0, m->stream, m->params, dx, dy, n);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpyAsync(y, dy, (size_t)n * kMlpOut * sizeof(float), hipMemcpyDeviceToHost, m->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(m->stream);
    (void)hipFree(dx);
    if (dy) (void)hipFree(dy);
    if (e != hipSuccess) return lbm_fail(LBM_ERR_HIP, "network forward: %s", hipGetErrorString(e));
    return LBM_OK;
}

int lbm_mlp_forward(lbm_mlp* m, const float* x, int n, float* y)
{
    return mlp_forward_impl(m, x, n, y, LBM_MLP_F32);
}

int lbm_mlp_forward_bf16(lbm_mlp* m, const float* x, int n, float* y)
{
    return mlp_forward_impl(m, x, n, y, LBM_MLP_BF16);
}

int lbm_mlp_forward_f16(lbm_mlp* m, const float* x, int n, float* y)
{
    return mlp_forward_impl(m, x, n, y, LBM_MLP_F16);
}

int lbm_mlp_loss_grad(lbm_mlp* m, const float* x, const float* t, int n, float* grad, double* loss)
{
    int rc = mlp_check(m);
    if (rc) return rc;
    if (!x || !t || n < 1) return lbm_fail(LBM_ERR_INVALID, "bad arguments");
    float *dx = nullptr, *dt = nullptr;
    MLP_TRY(hipMalloc(&dx, (size_t)n * kMlpIn * sizeof(float)));
    hipError_t e = hipMalloc(&dt, (size_t)n * kMlpOut * sizeof(float));
    if (e == hipSuccess) e = hipMemcpyAsync(dx, x, (size_t)n * kMlpIn * sizeof(float), hipMemcpyHostToDevice, m->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(dt, t, (size_t)n * kMlpOut * sizeof(float), hipMemcpyHostToDevice, m->stream);
    if (e == hipSuccess) {
        rc = mlp_grad(m, dx, dt, n, n, 0, 0);
        if (rc != LBM_OK) e = hipErrorUnknown;
    }
    if (e == hipSuccess && grad)
        e = hipMemcpyAsync(grad, m->grad, kMlpParams * sizeof(float), hipMemcpyDeviceToHost, m->stream);
    if (e == hipSuccess && loss) e = hipMemcpyAsync(loss, m->loss, sizeof(double), hipMemcpyDeviceToHost, m->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(m->stream);
    (void)hipFree(dx);
    if (dt) (void)hipFree(dt);
    if (rc != LBM_OK) return rc;
    if (e != hipSuccess) return lbm_fail(LBM_ERR_HIP, "network gradient: %s", hipGetErrorString(e));
    return LBM_OK;
}

}  // extern "C"

// ---------------------------------------------------------------------------
// Loss gradient without allocation (lbm_mlp_loss_grad_noalloc): the staged
// samples, the per-block partials, the gradient and the loss live in one
// file-scope device array, `scratch`, of fixed size (every device the
// library runs on holds its own copy until the process ends).  Its device
// address is looked up once per device with hipGetSymbolAddress; host code
// passes that address, never the array's name, to copies and kernels.
// Every call on one device shares the array: overlapping calls race.
// Nothing in it needs clearing: each block writes its whole partial, and
// the reduction writes the gradient and the loss.
// ---------------------------------------------------------------------------
namespace {

constexpr int kNoAllocSamples = 16384;
constexpr int kNoAllocBlocks = kGradBlocks;  // partials
constexpr size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }
constexpr size_t kScrPartial = 0;
constexpr size_t kScrLossPart = kScrPartial + align256((size_t)kNoAllocBlocks * kMlpParams * sizeof(float));
constexpr size_t kScrGrad = kScrLossPart + align256((size_t)kNoAllocBlocks * sizeof(double));
constexpr size_t kScrLoss = kScrGrad + align256((size_t)kMlpParams * sizeof(float));
constexpr size_t kScrX = kScrLoss + align256(sizeof(double));
constexpr size_t kScrT = kScrX + align256((size_t)kNoAllocSamples * kMlpIn * sizeof(float));
constexpr size_t kScratchBytes = kScrT + align256((size_t)kNoAllocSamples * kMlpOut * sizeof(float));  // 6.7 MB

static __device__ __align__(256) unsigned char scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
unsigned char* g_scratch_ptr[kMaxDevices] = {};

// Device address of `scratch` on device `dev` (which must be current).
int scratch_address(int dev, unsigned char** out)
{
    if (dev < 0 || dev >= kMaxDevices) return lbm_fail(LBM_ERR_INVALID, "device %d beyond %d", dev, kMaxDevices);
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return lbm_fail(LBM_ERR_HIP, "hipGetSymbolAddress(scratch) on device %d: %s", dev, hipGetErrorString(e));
        g_scratch_ptr[dev] = static_cast<unsigned char*>(p);
    }
    *out = g_scratch_ptr[dev];
    return LBM_OK;
}

}  // namespace

extern "C" {

int lbm_mlp_loss_grad_noalloc(lbm_mlp* m, const float* x, const float* t, int n, float* grad, double* loss)
{
    int rc = mlp_check(m);
    if (rc) return rc;
    if (!x || !t || n < 1) return lbm_fail(LBM_ERR_INVALID, "bad arguments");
    if (n > kNoAllocSamples)
        return lbm_fail(LBM_ERR_INVALID, "%d samples exceed the %d that lbm_mlp_loss_grad_noalloc holds", n,
                        kNoAllocSamples);
    unsigned char* base = nullptr;
    if ((rc = scratch_address(m->dev, &base))) return rc;
    float* dx = reinterpret_cast<float*>(base + kScrX);
    float* dt = reinterpret_cast<float*>(base + kScrT);
    float* partial = reinterpret_cast<float*>(base + kScrPartial);
    double* loss_part = reinterpret_cast<double*>(base + kScrLossPart);
    float* dgrad = reinterpret_cast<float*>(base + kScrGrad);
    double* dloss = reinterpret_cast<double*>(base + kScrLoss);
    // the same launch shape as lbm_mlp_loss_grad, so the sums run in the
    // same order and the results are the same bits
    const int nb = mlp_grad_blocks(n);
    MLP_TRY(hipMemcpyAsync(dx, x, (size_t)n * kMlpIn * sizeof(float), hipMemcpyHostToDevice, m->stream));
    MLP_TRY(hipMemcpyAsync(dt, t, (size_t)n * kMlpOut * sizeof(float), hipMemcpyHostToDevice, m->stream));
    hipLaunchKernelGGL(k_mlp_grad_partial, dim3(nb), dim3(kGradThreads), 0, m->stream, m->params, dx, dt, n, n,
                       (uint64_t)0, 0, partial, loss_part);
    MLP_TRY(hipGetLastError());
    hipLaunchKernelGGL(k_mlp_grad_reduce, dim3((kMlpParams + 63) / 64), dim3(1024), 0, m->stream, partial, nb,
                       dgrad, loss_part, dloss, n);
    MLP_TRY(hipGetLastError());
    if (grad) MLP_TRY(hipMemcpyAsync(grad, dgrad, kMlpParams * sizeof(float), hipMemcpyDeviceToHost, m->stream));
    if (loss) MLP_TRY(hipMemcpyAsync(loss, dloss, sizeof(double), hipMemcpyDeviceToHost, m->stream));
    MLP_TRY(hipStreamSynchronize(m->stream));
    return LBM_OK;
}

int lbm_mlp_clear_samples(lbm_mlp* m)
{
    if (!m) return lbm_fail(LBM_ERR_INVALID, "null network");
    m->samples = 0;
    return LBM_OK;
}

int lbm_mlp_normalize_samples(lbm_mlp* m, float* in_rms, float* out_rms)
{
    int rc = mlp_check(m);
    if (rc) return rc;
    if (m->samples < 1) return lbm_fail(LBM_ERR_INVALID, "no samples to normalize");
    constexpr int kBlocks = 256;
    double* part = nullptr;
    MLP_TRY(hipMalloc(&part, 2 * kBlocks * sizeof(double)));
    const size_t nx = (size_t)m->samples * kMlpIn, nt = (size_t)m->samples * kMlpOut;
    hipLaunchKernelGGL(k_sumsq, dim3(kBlocks), dim3(256), 0, m->stream, m->X, nx, part);
    hipLaunchKernelGGL(k_sumsq, dim3(kBlocks), dim3(256), 0, m->stream, m->T, nt, part + kBlocks);
    double host[2 * kBlocks];
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpyAsync(host, part, sizeof host, hipMemcpyDeviceToHost, m->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(m->stream);
    (void)hipFree(part);
    if (e != hipSuccess) return lbm_fail(LBM_ERR_HIP, "sample statistics: %s", hipGetErrorString(e));
    double sx = 0.0, st = 0.0;
    for (int b = 0; b < kBlocks; ++b) {
        sx += host[b];
        st += host[kBlocks + b];
    }
    const float rx = (float)std::sqrt(sx / (double)nx), rt = (float)std::sqrt(st / (double)nt);
    if (!(rx > 0.0f) || !(rt > 0.0f) || !std::isfinite(rx) || !std::isfinite(rt))
        return lbm_fail(LBM_ERR_INVALID, "samples have zero or non-finite spread");
    hipLaunchKernelGGL(k_scale, dim3(kBlocks), dim3(256), 0, m->stream, m->X, nx, 1.0f / rx);
    hipLaunchKernelGGL(k_scale, dim3(kBlocks), dim3(256), 0, m->stream, m->T, nt, 1.0f / rt);
    MLP_TRY(hipGetLastError());
    MLP_TRY(hipStreamSynchronize(m->stream));
    m->s_in *= rx;
    m->s_out *= rt;
    ++m->generation;
    if (in_rms) *in_rms = rx;
    if (out_rms) *out_rms = rt;
    return LBM_OK;
}

int lbm_mlp_sample_count(lbm_mlp* m, int* n)
{
    if (!m || !n) return lbm_fail(LBM_ERR_INVALID, "null argument");
    *n = m->samples;
    return LBM_OK;
}

int lbm_mlp_read_samples(lbm_mlp* m, int offset, int count, float* x, float* t)
{
    int rc = mlp_check(m);
    if (rc) return rc;
    if (offset < 0 || count < 0 || offset > m->samples || count > m->samples - offset)
        return lbm_fail(LBM_ERR_INVALID, "samples [%d, %d) outside the %d stored", offset, offset + count, m->samples);
    if (count == 0) return LBM_OK;
    if (x)
        MLP_TRY(hipMemcpyAsync(x, m->X + (size_t)offset * kMlpIn, (size_t)count * kMlpIn * sizeof(float),
                               hipMemcpyDeviceToHost, m->stream));
    if (t)
        MLP_TRY(hipMemcpyAsync(t, m->T + (size_t)offset * kMlpOut, (size_t)count * kMlpOut * sizeof(float),
                               hipMemcpyDeviceToHost, m->stream));
    MLP_TRY(hipStreamSynchronize(m->stream));
    return LBM_OK;
}

int lbm_mlp_add_samples(lbm_mlp* m, const float* x, const float* t, int n)
{
    int rc = mlp_check(m);
    if (rc) return rc;
    if (!x || !t || n < 0 || m->samples + n > m->capacity)
        return lbm_fail(LBM_ERR_INVALID, "samples exceed the capacity of %d", m->capacity);
    MLP_TRY(hipMemcpyAsync(m->X + (size_t)m->samples * kMlpIn, x, (size_t)n * kMlpIn * sizeof(float),
                           hipMemcpyHostToDevice, m->stream));
    MLP_TRY(hipMemcpyAsync(m->T + (size_t)m->samples * kMlpOut, t, (size_t)n * kMlpOut * sizeof(float),
                           hipMemcpyHostToDevice, m->stream));
    MLP_TRY(hipStreamSynchronize(m->stream));
    m->samples += n;
    return LBM_OK;
}

int lbm_mlp_add_transition(lbm_mlp* m, const float* state_t, const float* state_t1, const uint8_t* solid, int nx,
                           int ny, float tau, float force_x, float force_y, int stride, int offset, int* added)
{
    int rc = mlp_check(m);
    if (rc) return rc;
    if (!state_t || !state_t1 || !solid || nx < 3 || ny < 3 || stride < 1 || offset < 0 || !(tau > 0.5f))
        return lbm_fail(LBM_ERR_INVALID, "bad arguments");
    const size_t n = (size_t)nx * (size_t)ny;
    float *s0 = nullptr, *s1 = nullptr;
    uint8_t* sd = nullptr;
    MLP_TRY(hipMalloc(&s0, 9 * n * sizeof(float)));
    hipError_t e = hipMalloc(&s1, 9 * n * sizeof(float));
    if (e == hipSuccess) e = hipMalloc(&sd, n);
    if (e == hipSuccess) e = hipMemcpyAsync(s0, state_t, 9 * n * sizeof(float), hipMemcpyHostToDevice, m->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(s1, state_t1, 9 * n * sizeof(float), hipMemcpyHostToDevice, m->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(sd, solid, n, hipMemcpyHostToDevice, m->stream);
    const size_t cand = (n - (size_t)std::min<int>(offset, (int)n) + stride - 1) / stride;
    const size_t nblk = (cand + 255) / 256;
    int* blk = nullptr;  // per-block counts, then per-block first slots
    std::vector<int> base(nblk);
    int64_t total = m->samples;
    if (e == hipSuccess && nblk > 0) e = hipMalloc(&blk, nblk * sizeof(int));
    if (e == hipSuccess && nblk > 0) {
        hipLaunchKernelGGL(k_mlp_transition_count, dim3((unsigned)nblk), dim3(256), 0, m->stream, sd, nx, ny,
                           (uint32_t)stride, (uint32_t)offset, blk);
        e = hipGetLastError();
        if (e == hipSuccess) e = hipMemcpyAsync(base.data(), blk, nblk * sizeof(int), hipMemcpyDeviceToHost, m->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(m->stream);
        if (e == hipSuccess) {
            // exclusive scan from the running count; bases past the capacity
            // are clamped (those blocks store nothing)
            for (size_t b = 0; b < nblk; ++b) {
                const int cnt = base[b];
                base[b] = (int)std::min<int64_t>(total, m->capacity);
                total += cnt;
            }
            e = hipMemcpyAsync(blk, base.data(), nblk * sizeof(int), hipMemcpyHostToDevice, m->stream);
        }
        if (e == hipSuccess) {
            PhysArgs pa{};
            pa.nx = nx;
            pa.ny = ny;
            pa.omega = 1.0f / tau;
            pa.gx = force_x;
            pa.gy = force_y;
            pa.scale = pa.inv_scale = 1.0f;
            set_force_terms(pa);
            hipLaunchKernelGGL(k_mlp_transition, dim3((unsigned)nblk), dim3(256), 0, m->stream, s0, s1, sd, pa,
                               m->s_in, m->s_out, (uint32_t)stride, (uint32_t)offset, m->capacity, blk, m->X, m->T);
            e = hipGetLastError();
        }
    }
    if (e == hipSuccess) e = hipStreamSynchronize(m->stream);
    (void)hipFree(s0);
    if (s1) (void)hipFree(s1);
    if (sd) (void)hipFree(sd);
    if (blk) (void)hipFree(blk);
    if (e != hipSuccess) return lbm_fail(LBM_ERR_HIP, "transition samples: %s", hipGetErrorString(e));
    total = std::min<int64_t>(total, m->capacity);
    if (added) *added = (int)(total - m->samples);
    m->samples = (int)total;
    return LBM_OK;
}

int lbm_mlp_train(lbm_mlp* m, int steps, int batch, float lr, uint64_t seed, double* last_loss)
{
    int rc = mlp_check(m);
    if (rc) return rc;
    if (steps < 0 || batch < 1 || !(lr > 0.0f)) return lbm_fail(LBM_ERR_INVALID, "bad arguments");
    if (m->samples < 1) return lbm_fail(LBM_ERR_INVALID, "no samples to train on");
    if ((rc = mlp_quiesce_device(m))) return rc;
    ++m->generation;
    const double b1 = 0.9, b2 = 0.999, eps = 1e-8;
    for (int s = 0; s < steps; ++s) {
        rc = mlp_grad(m, m->X, m->T, m->samples, batch, seed + 0xD1B54A32D192ED03ull * (uint64_t)(m->adam_step + 1), 1);
        if (rc != LBM_OK) return rc;
        ++m->adam_step;
        const double c1 = 1.0 - std::pow(b1, (double)m->adam_step);
        const double c2 = 1.0 - std::pow(b2, (double)m->adam_step);
        hipLaunchKernelGGL(k_mlp_adam, dim3((kMlpParams + 255) / 256), dim3(256), 0, m->stream, m->params, m->grad,
                           m->adam_m, m->adam_v, (double)lr, b1, b2, eps, c1, c2);
        MLP_TRY(hipGetLastError());
    }
    if ((rc = mlp_repack(m))) return rc;
    if (last_loss) MLP_TRY(hipMemcpyAsync(last_loss, m->loss, sizeof(double), hipMemcpyDeviceToHost, m->stream));
    MLP_TRY(hipStreamSynchronize(m->stream));
    return LBM_OK;
}

}  // extern "C"
