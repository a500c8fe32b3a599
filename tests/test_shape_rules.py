"""Rules that pick a kernel shape from sizes alone, evaluated by the compiler."""
import subprocess

from simuverse_amd import build as B


def holds(tmp_path, *conditions):
    src = tmp_path / "rule.hip"
    src.write_text('#include "lbm_internal.hpp"\n' + "".join(f"static_assert({c});\n" for c in conditions))
    r = subprocess.run([B.hipcc(), "--offload-arch=gfx950", "-std=c++17", "--cuda-host-only", "-fsyntax-only", "-I",
                        str(B.ROOT / "include"), "-I", str(B.CSRC), str(src)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr


def test_d3q19_default_stores(tmp_path):
    """Plain stores (1) only where they measured faster than non-temporal ones
    (0): buffers of (nx, ny, nz, element bytes) in both storages."""
    cells = {(32, 32, 32, 4): 1, (40, 40, 40, 2): 1, (48, 48, 48, 4): 0, (36, 36, 36, 4): 0, (52, 52, 52, 4): 0,
             (64, 64, 64, 2): 0, (256, 256, 3, 4): 0, (60, 60, 60, 2): 0, (16, 128, 48, 2): 0, (56, 56, 56, 4): 1,
             (64, 64, 64, 4): 1, (72, 72, 72, 2): 1, (128, 128, 100, 4): 1, (200, 144, 90, 2): 1, (200, 144, 90, 4): 0,
             (256, 256, 256, 2): 0, (3, 3, 3, 4): 1}
    holds(tmp_path, *(f"lbm::default_variant3({2 * 19 * ((nx + 15) // 16 * 16) * ny * nz * e}ull) == {v}"
                      for (nx, ny, nz, e), v in cells.items()))
