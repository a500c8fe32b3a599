"""Properties of the gfx950 code the compiler makes of a kernel, read from its
assembly listing: they show here, without a GPU, what a timing would."""
import re
import subprocess

import pytest

from simuverse_amd import build as B


@pytest.fixture(scope="module")
def listing(tmp_path_factory):
    """Kernel name -> instructions, of one source file."""
    done = {}

    def get(src):
        if src not in done:
            out = tmp_path_factory.mktemp("asm") / (src + ".s")
            subprocess.run([B.hipcc(), *B.HIPCC_FLAGS, "-w", *B.EXTRA_FLAGS.get(src, []), "-I", str(B.ROOT / "include"),
                            "-I", str(B.CSRC), "--cuda-device-only", "-S", str(B.CSRC / src), "-o", str(out)],
                           check=True, capture_output=True, timeout=600)
            done[src] = {m.group(1): [t.split()[0] for t in (x.split(";")[0].strip() for x in m.group(2).split("\n"))
                                      if re.match(r"[a-z]\w+_", t)]
                         for m in re.finditer(r"^(_Z\S+):\s*; @.*?\n(.*?)\.Lfunc_end", out.read_text(), re.S | re.M)}
        return done[src]

    return get


@pytest.mark.parametrize("elem", ["f", "DF16_"], ids=["f32", "f16"])
def test_forced_d3q19_step_loads_its_constants_side_by_side(listing, elem):
    """Arguments and 41 force constants in a few wide scalar loads: twice as
    many loads cost 3 to 7 % of a step."""
    kernels = {k: v for k, v in listing("lbm3d.hip").items() if f"k3_stepI{elem}Lb1ELi" in k}
    assert len(kernels) >= 8
    for name, code in kernels.items():
        loads = sum(op.startswith("s_load") for op in code)
        assert loads <= 16, f"{name}: {loads} scalar loads"
