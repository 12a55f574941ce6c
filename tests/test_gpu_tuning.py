"""What the read-back of shape and form says of automatic runs, and that a
context set to it, or tuned, walks as one left alone: bit-exact walkers, echo
sums to 1e-12."""
import numpy as np
import pytest

import randomwalk_nmr_amd as R

pytestmark = pytest.mark.gpu

RTOL = 1e-12


def _inputs(dims, n, seed):
    W, H, D = dims
    rng = np.random.default_rng(seed)
    solid = (rng.random((D, H, W)) < 0.3).astype(np.uint8)
    w = R.setup_walkers(solid, seed, n)
    return solid, w["x"], w["y"], w["z"], w["seed"]


def _same(g, o):
    for k in ("x", "y", "z", "seed", "hits", "energy"):
        assert np.array_equal(g[k], o[k]), k
    assert np.all(np.abs(g["echo_sums"] - o["echo_sums"]) <= RTOL * o["echo_sums"])


# the lines of the automatic choice (sorted from about 2 ms of walk on)
@pytest.mark.parametrize("n,spe,shape,form", [(2000, 3, (64, 1), 5), (49_152, 3, (64, 1), 5), (65_536, 3, (64, 1), 5),
                                              (65_537, 3, (256, 1), 6), (524_288, 1250, (1024, 1), 6)])
def test_read_back_tells_what_ran_and_repeats_it(n, spe, shape, form):
    print(f"[test] read-back n={n} spe={spe}", flush=True)
    solid, *w = _inputs((40, 32, 24), n, 9)
    kw = dict(echoes=4, steps_per_echo=spe, bc="mirror", delta=0.995)
    with R.Context(0) as ctx:
        img = R.Image.from_solid(ctx, solid)
        assert ctx.get_launch() == (256, 1) and ctx.get_tuning()[:3] == (256, 1, 3)
        g = R.cpmg_run(ctx, img, *w, **kw)
        t = ctx.get_tuning()
        assert t[:2] == ctx.get_launch() == shape and t[2] == form
        img.close()
    with R.Context(0) as ctx:
        ctx.set_launch(*t[:2])
        ctx.set_unfolded(t[2])
        img = R.Image.from_solid(ctx, solid)
        _same(R.cpmg_run(ctx, img, *w, **kw), g)
        assert ctx.get_tuning()[:3] == t[:3]
        img.close()


def test_read_back_of_settings():
    """Settings are reported as set, whatever ran before."""
    print("[test] read-back of settings", flush=True)
    solid, *w = _inputs((32, 32, 32), 500, 2)
    with R.Context(0) as ctx:
        img = R.Image.from_solid(ctx, solid)
        R.cpmg_run(ctx, img, *w, echoes=2, steps_per_echo=3, bc="mirror", delta=0.995)
        ctx.set_launch(128, 2)
        assert ctx.get_launch() == (128, 2)
        ctx.set_unfolded(4)
        R.map_run(ctx, img, *w, steps=5, bc="mirror")
        assert ctx.get_tuning()[:3] == (128, 2, 4)
        ctx.set_launch(0, 0)
        assert ctx.get_launch() == (256, 1)
        img.close()


@pytest.mark.parametrize("bc", ["noflux", "periodic", "mirror"])
@pytest.mark.parametrize("n", [3000, 70_000])
def test_tuned_context_walks_runs_of_other_sizes(bc, n):
    """Tuned for n walkers, then runs of n, of few and of many: as a context
    left alone.  Short runs of many walkers are not sorted by the tuning."""
    print(f"[test] tuned, other sizes bc={bc} n={n}", flush=True)
    solid, *w = _inputs((48, 40, 32), 90_000, 5)
    kw = dict(echoes=6, steps_per_echo=5, bc=bc, delta=0.995)
    out = []
    for tuned in (False, True):
        with R.Context(0) as ctx:
            img = R.Image.from_solid(ctx, solid)
            if tuned:
                tpb, k, ms = ctx.autotune(img, *(a[:n] for a in w), steps_per_echo=5, bc=bc, trial_echoes=30,
                                          delta=0.995)
                t = ctx.get_tuning()
                assert t[:2] == (tpb, k) and ms > 0
                # every form that the library takes by itself here is a candidate
                assert t[2] in ((0, 3, 5, 6) if n <= 65_536 else (0, 3, 6))
            out.append([R.cpmg_run(ctx, img, *(a[:m] for a in w), **kw) for m in (n, 500, 90_000)])
            img.close()
    for g, o in zip(out[1], out[0]):
        _same(g, o)


def test_tuning_keeps_what_was_asked_for():
    """A form and a shape set by the caller leave nothing automatic to return to."""
    print("[test] tuned, form and shape set", flush=True)
    solid, *w = _inputs((32, 32, 32), 2000, 6)
    with R.Context(0) as ctx:
        img = R.Image.from_solid(ctx, solid)
        ctx.set_unfolded(0)
        ctx.set_launch(512, 1)
        tpb, k, _ = ctx.autotune(img, *w, steps_per_echo=3, bc="mirror", trial_echoes=20, delta=0.995)
        assert ctx.get_tuning()[:3] == (tpb, k, 0)
        img.close()
