"""Labelled, label-set and Jacobian walks on every unfolded image kind (noflux,
periodic and mirror, sides that are powers of two or not) against the oracle,
over more steps than a packed displacement holds: walkers, energies and hits
bit for bit, sums to 1e-12."""
import math

import numpy as np
import pytest

import oracle as O
import randomwalk_nmr_amd as R

pytestmark = pytest.mark.gpu

RTOL = 1e-12


@pytest.mark.parametrize("bc", ["noflux", "periodic", "mirror"])
@pytest.mark.parametrize("dims", [(32, 32, 32), (30, 21, 17), (128, 160, 130), (128, 128, 128)])
@pytest.mark.parametrize("echoes,spe", [(4, 257), (5, 102)])
def test_label_walks_match_oracle(bc, dims, echoes, spe):
    print(f"[test] label walks bc={bc} dims={dims} echoes={echoes} x {spe}", flush=True)
    W, H, D = dims
    rng = np.random.default_rng(W + spe)
    solid = (rng.random((D, H, W)) < 0.3).astype(np.uint8)
    labels = R.voronoi_labels(solid, 12, 8, 4)
    w = R.setup_walkers(solid, 7, 700)
    walk = (w["x"], w["y"], w["z"], w["seed"])
    # small penalties: energies stay within a few orders of magnitude over the run
    delta = 1.0 - np.linspace(1e-4, 2e-3, 8)
    sets = np.stack([delta, 1.0 - (1.0 - delta[::-1]) / 2])
    kw = dict(echoes=echoes, steps_per_echo=spe, bc=bc)
    with R.Context(0) as ctx:
        img = R.Image.from_solid(ctx, solid, labels=labels, n_labels=8)
        g = R.cpmg_run(ctx, img, *walk, label_delta=delta, label_hits=True, **kw)
        s = R.cpmg_run_label_sets(ctx, img, *walk, set_label_delta=sets, **kw)
        j = R.cpmg_forward_jacobian(ctx, img, *walk, label_delta=delta,
                                    label_hits=np.zeros((8, len(w["x"])), np.uint32), **kw)
        img.close()
    blocks = O.bitblock_pack(solid)
    o = O.walk(blocks, dims, *walk, labels=labels, label_delta=delta, label_hits=True, **kw)
    o1 = O.walk(blocks, dims, *walk, labels=labels, label_delta=sets[1], **kw)
    for r in (g, s, j):
        for k in ("x", "y", "z", "seed"):
            assert np.array_equal(r[k], o[k]), k
        assert np.array_equal(r["energy"].view(np.uint64), o["energy"].view(np.uint64))
    assert np.array_equal(g["hits"], o["hits"])
    for r in (g, j):
        assert np.array_equal(r["label_hits"].T, o["label_hits"])
        assert np.all(np.abs(r["echo_sums"] - o["echo_sums"]) <= RTOL * o["echo_sums"])
    for q, ref in enumerate((o, o1)):
        assert np.all(np.abs(s["echo_sums"][q] - ref["echo_sums"]) <= RTOL * ref["echo_sums"])
    ref = np.array([math.fsum(o["energy"] * o["label_hits"][:, l]) for l in range(8)])
    assert np.all(np.abs(j["jac"][:, -1] - ref) <= RTOL * np.abs(ref).max())
