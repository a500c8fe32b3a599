"""The build refuses step kernels whose vector registers go through scratch
memory: read from the compiler's remarks on two small kernels."""
import subprocess

from simuverse_amd import build as B

SOURCE = """
#include <hip/hip_runtime.h>
// more live values than the 64 registers of eight waves per SIMD
__global__ __launch_bounds__(1024, 8) void k_spills(const float* __restrict__ a, float* __restrict__ b)
{
    float v[100];
#pragma unroll
    for (int i = 0; i < 100; ++i) {
        v[i] = a[threadIdx.x + 1024 * i];
        asm volatile("" : "+v"(v[i]));
    }
    __syncthreads();
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < 100; ++i) s = s * v[i] + v[99 - i];
    b[threadIdx.x] = s;
}
__global__ void k_clean(float* b) { b[threadIdx.x] *= 2.0f; }
"""


def test_scratch_users_are_named(tmp_path):
    src = tmp_path / "k.hip"
    src.write_text(SOURCE)
    r = subprocess.run([B.hipcc(), *B.HIPCC_FLAGS, "-Rpass-analysis=kernel-resource-usage", "-c", str(src), "-o",
                        str(tmp_path / "k.o")], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    named = B.scratch_users(r.stderr)
    assert len(named) == 1 and "k_spills" in named[0]


def test_every_step_kernel_source_is_looked_at():
    assert B.NO_SCRATCH <= set(B.SOURCES)
    for src in B.SOURCES:
        text = (B.CSRC / src).read_text()
        assert ("__launch_bounds__" not in text) or src in B.NO_SCRATCH | {"lbm_learned.hip", "lbm_mlp.hip"}, src
