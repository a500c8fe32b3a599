"""The N-step shapes and the rule that picks one where the caller did not.

Every N-step shape equals the one-step shapes bit for bit through the
variant tests; here the rule's choice is compared with one launch per step
at every slot of both buffers, at sizes on its lines and at the edges of the
tiles.
"""
import numpy as np
import pytest

from simuverse_amd import lbm as L
from simuverse_amd import workloads as W

pytestmark = pytest.mark.gpu

# (nx, ny, x_edge): the smallest that fit nine steps, and five, below them one
# step; one tile and one cell more; 256 tiles of
# 16 x 16 and one column of tiles more; just above 2048 tiles of 24 x 24; and
# channels whose last tile would hold a single column of one or two shapes.
SIZES = [(9, 9, 0), (10, 12, 1), (5, 9, 1), (8, 30, 0), (4, 40, 0), (16, 16, 0), (17, 33, 1), (17, 17, 0),
         (256, 256, 1), (257, 256, 0), (1200, 1000, 1), (1177, 1100, 1), (1009, 1152, 1)]


def scene(nx, ny, x_edge):
    solid = np.zeros((ny, nx), bool)
    y, x = np.mgrid[0:ny, 0:nx]
    if x_edge:
        solid[[0, -1], :] = True
        spots = [(nx // 3, ny // 2, 4), (nx - 3, ny // 3, 3), (1, 2 * ny // 3, 2)]
    else:
        spots = [(0, ny // 2, 2), (nx // 2, 0, 1)]
    for cx, cy, r in spots:
        r = min(r, min(nx, ny) // 5)
        solid |= (x - cx) ** 2 + (y - cy) ** 2 <= r * r
    return solid


@pytest.mark.parametrize("layout", [L.LAYOUT_ROWS, L.LAYOUT_PLANES], ids=["rows", "planes"])
@pytest.mark.parametrize("storage", [L.STORAGE_F32, L.STORAGE_F16_DEV], ids=["f32", "f16"])
@pytest.mark.parametrize("nx, ny, x_edge", SIZES)
def test_default_shape_leaves_both_buffers_as_single_steps(nx, ny, x_edge, storage, layout):
    print(f"case: default shape {nx}x{ny} x_edge {x_edge} storage {storage} layout {layout}", flush=True)
    solid = scene(nx, ny, x_edge)
    kw = dict(x_edge=L.X_INLET_OUTLET, inlet_ux=0.05) if x_edge else dict(force=(1e-5, -2e-6))
    f0 = W.rest_state(nx, ny, solid, amplitude=1e-3).astype(np.float32)
    f0[:, solid] = 0.25  # solid slots no step writes keep what the caller wrote, buffer by buffer
    lats = []
    for fixed in (False, True):
        lat = L.Lattice(nx, ny, 0.58, storage=storage, layout=layout, **kw)
        lat.write_materials(W.materials_from_solid(solid))
        lat.write_populations(f0, 0)
        if fixed:
            lat.set_variant(lat.variant())  # as a caller's own choice: one step per launch
        lats.append(lat)
    assert lats[0].variant() == lats[1].variant()
    for steps in (1, 23, 100, 106, 205):
        for lat in lats:
            lat.run(steps)
        cur = lats[0].current_buffer()
        assert cur == lats[1].current_buffer()
        for buf in (cur, cur ^ 1):
            a, b = (lat.read_populations(buf) for lat in lats)
            assert np.array_equal(a, b, equal_nan=True), f"{steps} steps, buffer {buf - cur}: {np.count_nonzero(a != b)} slots differ"
    for lat in lats:  # the exported macro field of a last one-step launch
        lat.run(11, export_macro=True)
    for a, b in zip(lats[0].read_macro(), lats[1].read_macro()):
        assert np.array_equal(a, b, equal_nan=True)
    for lat in lats:
        lat.close()


@pytest.mark.parametrize("x_edge", [0, 1])
def test_set_variant_refuses_what_the_rule_refuses(x_edge):
    """lbm_set_variant and the Python mirror agree on the N-step shapes."""
    nstep = [v for v, s in enumerate(L.variant_shapes()) if s[3] & 256]
    assert len(nstep) >= 3
    for nx, ny in ((4, 30), (5, 5), (8, 9), (9, 9), (17, 20), (25, 20), (57, 20)):
        lat = L.Lattice(nx, ny, 0.6, x_edge=x_edge, inlet_ux=0.02 * x_edge)
        for v in nstep:
            if L.variant_ok(v, nx, ny, x_edge):
                lat.set_variant(v)
                assert lat.variant() == v
            else:
                with pytest.raises(Exception):
                    lat.set_variant(v)
        lat.close()
