"""The multi-step tiles' source run on the CPU (tests/cpp/emulated_hip stands
for the device language), under the address and bounds sanitizers: bits, stray
writes, reads out of range, values left in LDS, thread order, barriers.  The
asm statements are taken out: they are empty and only pin registers."""
import os
import re
import subprocess
from pathlib import Path

import pytest

from simuverse_amd import build as B

ROOT = Path(__file__).resolve().parent.parent
CPP = ROOT / "tests" / "cpp"
CLANG = Path("/opt/rocm/llvm/bin/clang++")


def plain(name):
    text = re.sub(r'asm volatile\(""[^;]*\);', "", (B.CSRC / name).read_text())
    assert "asm" not in re.sub(r"//.*", "", text), name
    return text


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("emulated")
    for name in ("lbm_cell.hpp", "lbm_device.hpp", "lbm_internal.hpp"):
        (d / name).write_text(plain(name))
    # the tile's body, without the kernels that call it and their launchers
    tile = plain("lbm_stepn.hip")
    end = tile.index("template <typename T, int XEDGE, bool FORCE, int BS, int RW, int RH, int NS, int FLAGS>\n// eight waves")
    (d / "lbm_stepn_tile.hpp").write_text(tile[:end] + "}\n")
    # the D3Q19 step kernels, without the kernels and the host code after them
    three = plain("lbm3d.hip")
    three = re.sub(r'#include "lbm(3d|_readback)\.(h|hpp)"\n', "", three)
    (d / "lbm3d_kernels.hpp").write_text(three[:three.index("// After a host write: slot k of each solid cell")] + "}\n}\n")

    def build(test):
        exe = d / test
        subprocess.run([str(CLANG), "-std=c++17", "-O1", "-g", "-mfma", "-mf16c", "-ffp-contract=off", "-Wno-unknown-pragmas",
                        "-Wno-pass-failed", "-fsanitize=address,array-bounds", "-fno-sanitize-recover=all", "-I",
                        str(CPP / "emulated_hip"), "-I", str(d), "-I", str(ROOT / "include"), str(CPP / (test + ".cpp")),
                        "-o", str(exe)], check=True, timeout=600)
        return exe

    return build


def run(exe, *args):
    r = subprocess.run([str(exe), *args], capture_output=True, text=True, timeout=600,
                       env=dict(os.environ, ASAN_OPTIONS="detect_leaks=0:detect_stack_use_after_return=0"))
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-3000:]
    return r.stdout


@pytest.fixture(scope="module")
def stepn(program):
    return program("test_stepn_emulated")


@pytest.mark.parametrize("shape", ["32x32x9", "32x32x5", "64x32x5", "64x48x5"])
def test_nstep_tiles(stepn, shape):
    assert f"{shape}: 0 bad" in run(stepn, shape)


def test_two_step_d3q19(program):
    assert "two steps: 0 bad" in run(program("test_step3d_emulated"))
