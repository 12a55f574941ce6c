"""Field walks in position order (large runs on fields that spill an XCD's L2)
against the caller's order: every walker bit for bit, echo sums to 1e-12 of
the walker count (the values of one echo lie within +-1 and are added in
another order)."""
import numpy as np
import pytest

import randomwalk_nmr_amd as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bc", ["noflux", "periodic", "mirror"])
@pytest.mark.parametrize("n,echoes", [(65_536, 32), (70_001, 33), (65_535, 32), (65_537, 31)])
def test_field_walk_in_position_order(bc, n, echoes):
    """Both sides of the walker and step counts that choose the order, with a
    re-sort between launches where it is taken."""
    print(f"[test] field order bc={bc} n={n} echoes={echoes}", flush=True)
    W, H, D = 101, 90, 75
    rng = np.random.default_rng(n)
    solid = (rng.random((D, H, W)) < 0.3).astype(np.uint8)
    field = rng.normal(size=(D, H, W))
    w = R.setup_walkers(solid, 3, n)
    pen = 1.0 - rng.uniform(0.001, 0.02, n)
    out = []
    for setting in ("default", "off", "resorted"):
        with R.Context(0) as ctx:
            if setting == "off":
                ctx.set_locality(False)
            elif setting == "resorted":
                ctx.set_locality(True, 10, 1)
            img = R.Image.from_solid(ctx, solid)
            out.append(R.cpmg_field_run(ctx, img, w["x"], w["y"], w["z"], w["seed"], echoes=echoes, steps_per_echo=8,
                                        field=field, gyromagnetic_ratio=42.576, time_interval_ms=0.01, bc=bc,
                                        penalty=pen))
            img.close()
    for o in out[1:]:
        for k in ("x", "y", "z", "seed", "hits", "p_alive", "phase", "energy"):
            assert np.array_equal(np.asarray(out[0][k]).view(np.uint8), np.asarray(o[k]).view(np.uint8)), k
        assert np.all(np.abs(out[0]["echo_sums"] - o["echo_sums"]) <= 1e-12 * n)


@pytest.mark.parametrize("bc", ["noflux", "periodic", "mirror"])
def test_no_walkers_in_position_order(bc):
    """A context that orders every run takes one without walkers: echo sums of 0."""
    print(f"[test] no walkers, ordered, bc={bc}", flush=True)
    rng = np.random.default_rng(1)
    solid = (rng.random((24, 32, 40)) < 0.3).astype(np.uint8)
    none = np.zeros(0, np.int32)
    w = (none, none, none, np.zeros(0, np.uint64))
    with R.Context(0) as ctx:
        ctx.set_locality(True, 10, 0)
        img = R.Image.from_solid(ctx, solid)
        f = R.cpmg_field_run(ctx, img, *w, echoes=25, steps_per_echo=4, field=rng.normal(size=solid.shape),
                             gyromagnetic_ratio=42.576, time_interval_ms=0.01, bc=bc)
        g = R.cpmg_run(ctx, img, *w, echoes=25, steps_per_echo=4, bc=bc)
        img.close()
    for o in (f, g):
        assert o["echo_sums"].shape == (26,) and not np.any(o["echo_sums"])
