"""Readbacks through the pinned slots: the same bytes whatever the size, into
fresh, reused and page-locked arrays."""
import numpy as np
import pytest
import torch

from simuverse_amd import lbm as L
from simuverse_amd import workloads as W

pytestmark = pytest.mark.gpu

# 12 n bytes of macro fields: under one slot of 1 MiB; pieces that straddle
# slots; two slots in turn; just under and from the 6 MiB on where four threads
# start; more chunks than slots; just under and over the 32 MiB where twelve do
SIZES = [(3, 3), (300, 291), (600, 375), (1024, 511), (1024, 512), (1531, 1037), (1700, 1644), (1700, 1650)]


@pytest.mark.parametrize("nx, ny", SIZES)
def test_macro_readback_bytes(nx, ny):
    print(f"case: readback {nx}x{ny}", flush=True)
    lat = L.Lattice(nx, ny, 0.7, force=(1e-6, 0.0))
    f = W.rest_state(nx, ny, np.zeros((ny, nx), bool), amplitude=1e-3).astype(np.float32)
    lat.write_populations(f, 0)
    lat.run(3)
    pop = lat.read_populations()
    assert np.array_equal(lat.read_populations(), pop)
    rho, ux, uy = lat.macro()
    # moments of the next gather have no simple form on the host; each field
    # alone and the three together must agree, in any destination
    lib = L.load_library()
    pinned = torch.empty((3, ny, nx), dtype=torch.float32, pin_memory=True).numpy()
    reused = np.full((3, ny, nx), np.nan, np.float32)
    for out in (pinned, reused, reused[::-1]):
        out[:] = np.nan
        p = [out[k].ctypes.data for k in range(3)]
        assert lib.lbm_macro(lat._h, *p) == 0
        for got, want in zip(out, (rho, ux, uy)):
            assert np.array_equal(got, want)
    for k, want in enumerate((rho, ux, uy)):
        one = np.full((ny, nx), np.nan, np.float32)
        p = [None, None, None]
        p[k] = one.ctypes.data
        assert lib.lbm_macro(lat._h, *p) == 0
        assert np.array_equal(one, want)
    edge = np.full((2, ny, nx), np.nan, np.float32)  # first and last: two runs
    assert lib.lbm_macro(lat._h, edge[0].ctypes.data, None, edge[1].ctypes.data) == 0
    assert np.array_equal(edge[0], rho) and np.array_equal(edge[1], uy)
    # the saved state holds the same populations
    other = L.Lattice(nx, ny, 0.7, force=(1e-6, 0.0))
    other.load_state(lat.save_state())
    assert np.array_equal(other.read_populations(other.current_buffer()), pop)
    lat.close()
    other.close()
