"""The readback's host side (simuverse_amd/csrc/lbm_readback.hpp) on the CPU,
against a stand-in for the runtime (tests/cpp/fake_hip), plain and under the
sanitizers."""
import os
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
CPP = ROOT / "tests" / "cpp"
BUILDS = {"plain": ["-O2"], "address": ["-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=all"],
          "thread": ["-O1", "-g", "-fsanitize=thread"]}


@pytest.fixture(scope="module", params=list(BUILDS))
def program(request, tmp_path_factory):
    exe = tmp_path_factory.mktemp("readback") / request.param
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Wextra", "-pthread", *BUILDS[request.param], "-I",
                    str(CPP / "fake_hip"), "-I", str(ROOT / "simuverse_amd" / "csrc"), str(CPP / "test_readback.cpp"),
                    "-o", str(exe)], check=True, timeout=300)
    return exe


@pytest.mark.parametrize("what", ["bytes", "one_chunk", "busy", "copy_fails", "pinned", "together", "short_of_memory"])
def test_readback(program, what):
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=1", TSAN_OPTIONS="halt_on_error=1")
    r = subprocess.run([str(program), what], capture_output=True, text=True, timeout=120, env=env)
    assert r.returncode == 0, r.stdout + r.stderr
    assert f"{what} ok" in r.stdout
