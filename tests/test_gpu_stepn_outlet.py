"""N-step tiles at the tightest width their rule admits: a channel whose last
tile holds two columns, so that the outlet column, which gathers as its west
neighbour, reads at the rim of the valid ring in every step.  338 leaves two
columns for tiles of 16, 24 and 56 columns alike; obstacles lie on the outlet
and inlet columns, and 72, 49 and 41 rows cut the tiles in y too."""
import numpy as np
import pytest

from simuverse_amd import lbm as L
from simuverse_amd import workloads as W

pytestmark = pytest.mark.gpu

NX = 338
BATCH_NX = 340  # a batch takes widths that are multiples of four: four columns are the fewest there
NSTEP = 256


def scene(nx, ny):
    y, x = np.mgrid[0:ny, 0:nx]
    solid = (y == 0) | (y == ny - 1)
    for cx, cy, r in ((nx - 1, ny // 4, 3), (nx - 2, ny // 2, 2), (nx - 4, 3 * ny // 4, 2), (0, ny // 3, 2),
                      (90, ny // 2, 5)):
        solid |= (x - cx) ** 2 + (y - cy) ** 2 <= r * r
    return solid, W.rest_state(nx, ny, solid, amplitude=1e-3).astype(np.float32)


def one_step(nx, ny, storage, layout, force, steps):
    solid, f0 = scene(nx, ny)
    lat = L.Lattice(nx, ny, 0.8, storage=storage, layout=layout, x_edge=L.X_INLET_OUTLET, inlet_ux=0.04, force=force)
    lat.write_materials(W.materials_from_solid(solid))
    lat.write_populations(f0, 0)
    lat.set_variant(lat.variant())  # one launch per step
    lat.run(steps)
    out = lat.read_populations()
    lat.close()
    assert np.isfinite(out[:, ~solid]).all()
    return solid, f0, out


@pytest.mark.parametrize("force", [(0.0, 0.0), (2e-6, -1e-6)], ids=["free", "force"])
@pytest.mark.parametrize("layout", [L.LAYOUT_ROWS, L.LAYOUT_PLANES], ids=["rows", "planes"])
@pytest.mark.parametrize("storage", [L.STORAGE_F32, L.STORAGE_F16_DEV], ids=["f32", "f16"])
@pytest.mark.parametrize("ny", [72, 49])
def test_two_column_last_tile(ny, storage, layout, force):
    print(f"case: {NX}x{ny} storage {storage} layout {layout} force {force}", flush=True)
    solid, f0, want = one_step(NX, ny, storage, layout, force, 203)
    shapes = L.variant_shapes()
    nstep = [v for v, s in enumerate(shapes) if s[3] & NSTEP]
    assert len(nstep) >= 4
    fl = ~solid
    for v in [None] + nstep:
        if v is not None:
            assert NX % shapes[v][2] == 2 and L.variant_ok(v, NX, ny, L.X_INLET_OUTLET)
        lat = L.Lattice(NX, ny, 0.8, storage=storage, layout=layout, x_edge=L.X_INLET_OUTLET, inlet_ux=0.04, force=force)
        lat.write_materials(W.materials_from_solid(solid))
        lat.write_populations(f0, 0)
        if v is not None:
            lat.set_variant(v)
        lat.run(203)
        got = lat.read_populations()
        lat.close()
        bad = np.count_nonzero(got[:, fl] != want[:, fl])
        assert bad == 0, f"shape {v} differs at {bad} slots of fluid cells"


@pytest.mark.parametrize("storage", [L.STORAGE_F32, L.STORAGE_F16_DEV], ids=["f32", "f16"])
def test_narrowest_last_tile_of_batched_domains(storage):
    print(f"case: batch of {BATCH_NX}-wide channels storage {storage}", flush=True)
    rows, forces, steps = (72, 49, 41), ((0.0, 0.0), (2e-6, -1e-6), (0.0, 0.0)), 138
    refs = [one_step(BATCH_NX, ny, storage, L.LAYOUT_ROWS, fo, steps) for ny, fo in zip(rows, forces)]
    shapes = L.batch_variant_shapes()
    nstep = [v for v, s in enumerate(shapes) if s[3] & NSTEP]
    assert len(nstep) >= 3
    for v in nstep:
        assert BATCH_NX % shapes[v][1] == 4
        b = L.Batch([dict(nx=BATCH_NX, ny=ny, tau=0.8, x_edge=L.X_INLET_OUTLET, inlet_ux=0.04, force=fo)
                     for ny, fo in zip(rows, forces)], storage=storage)
        for k, (solid, f0, _) in enumerate(refs):
            b.write_materials(k, W.materials_from_solid(solid))
            b.write_populations(k, f0)
        b.set_variant(v)
        b.run(steps)
        for k, (solid, _, want) in enumerate(refs):
            bad = np.count_nonzero(b.read_populations(k)[:, ~solid] != want[:, ~solid])
            assert bad == 0, f"batch shape {v}, domain {k}: {bad} slots of fluid cells differ"
        b.close()


@pytest.mark.parametrize("nx, ny, x_edge", [(9, 9, 0), (17, 33, 0), (40, 24, 1), (256, 120, 1), (1177, 300, 1)])
@pytest.mark.parametrize("storage", [L.STORAGE_F32, L.STORAGE_F16_DEV], ids=["f32", "f16"])
def test_default_shape_on_flows_that_stay_finite(nx, ny, x_edge, storage):
    """The rule's choice against one launch per step where every fluid slot is
    finite at the end, so that no comparison is of NaN with NaN."""
    print(f"case: default {nx}x{ny} x_edge {x_edge} storage {storage}", flush=True)
    y, x = np.mgrid[0:ny, 0:nx]
    solid = (x - nx // 2) ** 2 + (y - ny // 2) ** 2 <= 2
    if x_edge:
        solid |= (y == 0) | (y == ny - 1)
    f0 = W.rest_state(nx, ny, solid, amplitude=1e-3).astype(np.float32)
    kw = dict(x_edge=L.X_INLET_OUTLET, inlet_ux=0.03) if x_edge else dict(force=(1e-6, -2e-6))
    outs = []
    for fixed in (False, True):
        lat = L.Lattice(nx, ny, 0.9, storage=storage, **kw)
        lat.write_materials(W.materials_from_solid(solid))
        lat.write_populations(f0, 0)
        if fixed:
            lat.set_variant(lat.variant())
        lat.run(23)
        lat.run(412)
        cur = lat.current_buffer()
        outs.append([lat.read_populations(b) for b in (cur, cur ^ 1)])
        lat.close()
    fl = ~solid
    for a, b in zip(*outs):
        assert np.isfinite(b[:, fl]).all()
        assert np.array_equal(a[:, fl], b[:, fl])


@pytest.mark.parametrize("n, storage, variant", [(4096, L.STORAGE_F32, 50), (8192, L.STORAGE_F16_DEV, 51)],
                         ids=["4096-f32", "8192-f16"])
def test_full_size_five_step_shapes_match_one_step(n, storage, variant):
    """The two five-step shapes at the sizes the benchmark tunes to them for:
    35 steps and one more from the same seeded disks."""
    print(f"case: {n}x{n} shape {variant} against one step", flush=True)
    assert L.variant_shapes()[variant][3] & NSTEP
    sc = W.periodic_disks(n, n)
    outs = []
    for v in (6, variant):
        lat = L.Lattice(n, n, 0.55, force=(1e-6, 0.0), storage=storage)
        assert lat.variant() == 6
        lat.write_materials(W.materials_from_solid(sc.solid))
        lat.reset()
        lat.set_variant(v)
        lat.run(35)
        lat.run(1)
        outs.append(lat.read_populations())
        lat.close()
    for i in range(9):
        a, b = outs[0][i][~sc.solid], outs[1][i][~sc.solid]
        assert np.isfinite(a).all()
        assert np.array_equal(a, b), f"direction {i}: {np.count_nonzero(a != b)} slots differ"
