"""Host-array calls (walkers and results as one pinned block up to 4 MiB, array
by array above) against the same run on device arrays: every array bit for bit,
on both sides of the line, with and without the optional arrays, and after a
call that failed before or after its walkers were staged."""
import numpy as np
import pytest

import randomwalk_nmr_amd as R

pytestmark = pytest.mark.gpu


def _inputs(n):
    rng = np.random.default_rng(n)
    solid = (rng.random((24, 32, 40)) < 0.3).astype(np.uint8)
    return solid, R.setup_walkers(solid, 3, n), 1.0 - rng.uniform(0.001, 0.02, n)


# 32 bytes a walker, 40 with a penalty each: the line is at 131,072 and 104,857
@pytest.mark.parametrize("n", [1, 63, 64, 65, 2001, 104_800, 104_858, 131_072, 131_073])
@pytest.mark.parametrize("per_walker", [False, True])
def test_host_run_matches_device_run(n, per_walker):
    import torch

    print(f"[test] host staging n={n} per_walker={per_walker}", flush=True)
    solid, w, pen = _inputs(n)
    kw = dict(echoes=5, steps_per_echo=4, bc="mirror", penalty=pen if per_walker else None, delta=0.99)
    dev = lambda a, t: torch.from_numpy(a.copy()).to("cuda").view(t)
    with R.Context(0) as ctx:
        img = R.Image.from_solid(ctx, solid)
        g = R.cpmg_run(ctx, img, w["x"], w["y"], w["z"], w["seed"], **kw)
        m = R.map_run(ctx, img, w["x"], w["y"], w["z"], w["seed"], steps=20, bc="mirror")
        d = [dev(w[k], torch.int32) for k in "xyz"] + [dev(w["seed"].view(np.int64), torch.int64)]
        e = torch.ones(n, dtype=torch.float64, device="cuda")
        sums = torch.zeros(6, dtype=torch.float64, device="cuda")
        if per_walker:
            kw["penalty"] = dev(pen, torch.float64)
        R.cpmg_run(ctx, img, *d, energy=e, echo_sums=sums, **kw)
        img.close()
    for k, t in zip(("x", "y", "z", "seed"), d):
        assert np.array_equal(g[k].view(np.uint8), t.cpu().numpy().view(np.uint8)), k
        assert np.array_equal(g[k], m[k]), k
    assert np.array_equal(g["hits"], m["hits"])
    assert np.array_equal(g["energy"].view(np.uint64), e.cpu().numpy().view(np.uint64))
    assert np.array_equal(g["echo_sums"].view(np.uint64), sums.cpu().numpy().view(np.uint64))


def test_a_call_after_a_failed_one():
    """A walker outside a noflux image fails its call before anything is staged;
    the next is whole."""
    print("[test] host staging after an error", flush=True)
    solid, w, _ = _inputs(500)
    kw = dict(echoes=5, steps_per_echo=4, bc="noflux", delta=0.99)
    with R.Context(0) as ctx:
        img = R.Image.from_solid(ctx, solid)
        before = R.cpmg_run(ctx, img, w["x"], w["y"], w["z"], w["seed"], **kw)
        x = w["x"].copy()
        x[7] = 4000
        with pytest.raises(Exception):
            R.cpmg_run(ctx, img, x, w["y"], w["z"], w["seed"], **kw)
        after = R.cpmg_run(ctx, img, w["x"], w["y"], w["z"], w["seed"], **kw)
        img.close()
    for k in ("x", "y", "z", "seed", "hits", "energy", "echo_sums"):
        assert np.array_equal(before[k], after[k]), k


@pytest.mark.parametrize("n_failed", [300, 500, 40_000, 140_000])
@pytest.mark.parametrize("how", ["no field", "no unfolded image"])
def test_a_call_after_one_that_failed_once_staged(n_failed, how):
    """Refused with its walkers already copied in: its arrays stay as they were,
    also when later calls of fewer, as many and more walkers hand over theirs,
    and those calls are whole."""
    import ctypes as ct

    from randomwalk_nmr_amd._lib import load
    from randomwalk_nmr_amd.core import _ptr, _walker_struct, bc_code

    print(f"[test] host staging after a refusal once staged n={n_failed} {how}", flush=True)
    solid, w, _ = _inputs(500)
    kw = dict(echoes=5, steps_per_echo=4, bc="mirror", delta=0.99)
    labels = R.voronoi_labels(solid, 9, 8, 4)
    L = load()
    rng = np.random.default_rng(n_failed)
    bad = [rng.integers(0, 20, n_failed).astype(np.int32) for _ in range(3)]
    bad += [rng.integers(1, 1 << 62, n_failed).astype(np.uint64), rng.random(n_failed),
            rng.integers(0, 9, n_failed).astype(np.uint32), np.full(6, 7.0), np.full(48, 7.0)]
    kept = [a.copy() for a in bad]
    with R.Context(0) as ctx:
        img = R.Image.from_solid(ctx, solid, labels=labels, n_labels=8)
        before = R.cpmg_run(ctx, img, w["x"], w["y"], w["z"], w["seed"], **kw)
        st = _walker_struct(*bad[:4], bad[4], bad[5], None, 0.99, n_failed, 0)
        if how == "no field":
            code = L.rwnmr_cpmg_field_run(ctx.handle, img.handle, ct.byref(st), 5, 4, bc_code("mirror"), None, 42.0,
                                          0.1, None, None, _ptr(bad[6]))
        else:
            ctx.set_unfolded(0)
            delta = np.full(8, 0.99)
            code = L.rwnmr_cpmg_forward_jacobian(ctx.handle, img.handle, ct.byref(st), 5, 4, bc_code("mirror"),
                                                 _ptr(delta), None, _ptr(bad[6]), _ptr(bad[7]))
            ctx.set_unfolded(3)
        assert code != 0
        after = [R.cpmg_run(ctx, img, *(w[k][:m] for k in ("x", "y", "z", "seed")), **kw) for m in (500, 200, 500)]
        # more walkers than the refused call had
        big = R.setup_walkers(solid, 4, 60_000)
        R.cpmg_run(ctx, img, big["x"], big["y"], big["z"], big["seed"], **kw)
        after.append(R.cpmg_run(ctx, img, w["x"], w["y"], w["z"], w["seed"], **kw))
        img.close()
    for a, b in zip(bad, kept):
        assert np.array_equal(a, b)
    for g in after:
        m = len(g["x"])
        for k in ("x", "y", "z", "seed", "hits", "energy"):
            assert np.array_equal(g[k], before[k][:m]), k
        if m == 500:
            assert np.all(np.abs(g["echo_sums"] - before["echo_sums"]) <= 1e-12 * before["echo_sums"])
