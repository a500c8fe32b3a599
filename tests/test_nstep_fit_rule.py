"""Which lattices the N-step tile shapes admit (lbm.variant_ok, the library's
own rule): at least as many cells a side as steps, with the inlet/outlet edge a
last tile of two columns or more, rows and row stride below 2^24."""
from simuverse_amd import lbm as L


def test_nstep_fit_rule():
    shapes = L.variant_shapes()
    nstep = [v for v, s in enumerate(shapes) if s[3] & 256]
    assert len(nstep) >= 4
    for v in nstep:
        bw, steps = shapes[v][2], shapes[v][3] >> 12
        assert steps % 2 == 1  # launches flip the buffers as that many steps do
        assert L.variant_ok(v, steps, steps)
        assert not L.variant_ok(v, steps - 1, 64) and not L.variant_ok(v, 64, steps - 1)
        for tiles in (1, 2, 7):
            assert not L.variant_ok(v, tiles * bw + 1, 64, L.X_INLET_OUTLET)
            assert L.variant_ok(v, tiles * bw + 2, 64, L.X_INLET_OUTLET)
            assert L.variant_ok(v, tiles * bw + 1, 64, L.X_PERIODIC)
        assert L.variant_ok(v, steps, (1 << 24) - 1) and not L.variant_ok(v, steps, 1 << 24)
        big = (1 << 24) // 9 - 16
        assert L.variant_ok(v, big - 1, steps) and not L.variant_ok(v, big + 1, steps)
    batch = [s for s in L.batch_variant_shapes() if s[3] & 256]
    assert len(batch) >= 3 and all((s[3] >> 12) % 2 == 1 for s in batch)
