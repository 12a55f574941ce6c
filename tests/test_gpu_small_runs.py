"""Runs of few walkers (the speculative walk the library takes by itself) and
walks with voxel division on the unfolded image: bit-exact walkers and echo
sums to 1e-12 against the oracle, at the edges of echo groups, of odd and even
step counts, of the displacement flush and of the walker count that chooses
the form."""
import numpy as np
import pytest

import oracle as O
import randomwalk_nmr_amd as R

pytestmark = pytest.mark.gpu

RTOL = 1e-12


def _inputs(dims, n, seed, shift=0):
    W, H, D = dims
    rng = np.random.default_rng(seed)
    solid = (rng.random((D, H, W)) < 0.3).astype(np.uint8)
    w = R.setup_walkers(solid, seed, n, shift=shift)
    return solid, w["seed"], w["x"], w["y"], w["z"], 1.0 - rng.uniform(0.001, 0.02, n)


def _same(g, o, keys=("x", "y", "z", "seed", "hits")):
    for k in keys:
        assert np.array_equal(np.asarray(g[k]), np.asarray(o[k])), k


@pytest.mark.parametrize("bc", ["noflux", "periodic", "mirror"])
@pytest.mark.parametrize("dims", [(32, 32, 32), (30, 21, 17)])
@pytest.mark.parametrize("echoes,spe", [(1, 1), (7, 2), (8, 3), (17, 1), (33, 4), (5, 510), (4, 511), (3, 1023), (2, 0)])
def test_default_small_run_matches_oracle(bc, dims, echoes, spe):
    print(f"[test] small run bc={bc} dims={dims} echoes={echoes} x {spe}", flush=True)
    solid, seeds, x, y, z, pen = _inputs(dims, 777, 5 + spe)
    with R.Context(0) as ctx:
        img = R.Image.from_solid(ctx, solid)
        g = R.cpmg_run(ctx, img, x, y, z, seeds, echoes=echoes, steps_per_echo=spe, bc=bc, penalty=pen)
        m = R.map_run(ctx, img, x, y, z, seeds, steps=echoes * spe, bc=bc)
        img.close()
    o = O.walk(O.bitblock_pack(solid), dims, x, y, z, seeds, echoes=echoes, steps_per_echo=spe, bc=bc, penalty=pen)
    _same(g, o)
    _same(m, o)
    assert np.array_equal(g["energy"].view(np.uint64), o["energy"].view(np.uint64))
    assert np.all(np.abs(g["echo_sums"] - o["echo_sums"]) <= RTOL * o["echo_sums"])


@pytest.mark.parametrize("n", [1, 64, 65, 49_152, 49_153, 65_536, 65_537])
def test_walker_counts_that_choose_the_form(n):
    """Default context against the chunk-cache walk asked for by name."""
    print(f"[test] form choice n={n}", flush=True)
    solid, seeds, x, y, z, pen = _inputs((40, 32, 24), n, 9)
    out = []
    for asked in (False, True):
        with R.Context(0) as ctx:
            if asked:
                ctx.set_unfolded(3)
                ctx.set_launch(256, 1)
            img = R.Image.from_solid(ctx, solid)
            out.append(R.cpmg_run(ctx, img, x, y, z, seeds, echoes=21, steps_per_echo=5, bc="mirror", penalty=pen))
            img.close()
    _same(*out, keys=("x", "y", "z", "seed", "hits", "energy"))
    assert np.all(np.abs(out[0]["echo_sums"] - out[1]["echo_sums"]) <= RTOL * out[1]["echo_sums"])


@pytest.mark.parametrize("n", [49_152, 49_153])
@pytest.mark.parametrize("shift", [0, 1])
def test_walker_counts_that_choose_the_form_of_a_map(n, shift):
    print(f"[test] form choice of a map n={n} shift={shift}", flush=True)
    dims = (40, 32, 24)
    solid, seeds, x, y, z, _ = _inputs(dims, n, 9, shift)
    with R.Context(0) as ctx:
        img = R.Image.from_solid(ctx, solid)
        m = R.map_run(ctx, img, x, y, z, seeds, steps=101, bc="mirror", shift=shift)
        img.close()
    o = O.walk(O.bitblock_pack(solid), dims, x, y, z, seeds, echoes=1, steps_per_echo=101, bc="mirror", shift=shift)
    _same(m, o)


@pytest.mark.parametrize("threads", [64, 192, 1024])
def test_speculative_walk_sums_over_several_waves(threads):
    print(f"[test] speculative walk threads={threads}", flush=True)
    solid, seeds, x, y, z, pen = _inputs((30, 21, 17), 2500, 3)
    with R.Context(0) as ctx:
        ctx.set_unfolded(5)
        ctx.set_launch(threads, 1)
        img = R.Image.from_solid(ctx, solid)
        g = R.cpmg_run(ctx, img, x, y, z, seeds, echoes=43, steps_per_echo=3, bc="mirror", penalty=pen)
        img.close()
    o = O.walk(O.bitblock_pack(solid), (30, 21, 17), x, y, z, seeds, echoes=43, steps_per_echo=3, bc="mirror",
               penalty=pen)
    _same(g, o)
    assert np.all(np.abs(g["echo_sums"] - o["echo_sums"]) <= RTOL * o["echo_sums"])


@pytest.mark.parametrize("bc", ["noflux", "periodic", "mirror"])
@pytest.mark.parametrize("dims", [(16, 16, 16), (13, 9, 21), (2, 3, 64)])
@pytest.mark.parametrize("shift", [1, 2, 3])
@pytest.mark.parametrize("unfolded", [None, 3, 0])
def test_voxel_division_matches_oracle(bc, dims, shift, unfolded):
    """The speculative walk (default), the chunk-cache walk and the folded
    kernel with each voxel walked as 2^shift a side."""
    print(f"[test] divided bc={bc} dims={dims} shift={shift} form={unfolded}", flush=True)
    solid, seeds, x, y, z, pen = _inputs(dims, 900, 11, shift)
    with R.Context(0) as ctx:
        if unfolded is not None:
            ctx.set_unfolded(unfolded)
        img = R.Image.from_solid(ctx, solid)
        g = R.cpmg_run(ctx, img, x, y, z, seeds, echoes=19, steps_per_echo=31, bc=bc, shift=shift, penalty=pen)
        m = R.map_run(ctx, img, x, y, z, seeds, steps=19 * 31, bc=bc, shift=shift)
        img.close()
    o = O.walk(O.bitblock_pack(solid), dims, x, y, z, seeds, echoes=19, steps_per_echo=31, bc=bc, shift=shift,
               penalty=pen)
    _same(g, o)
    _same(m, o)
    assert np.array_equal(g["energy"].view(np.uint64), o["energy"].view(np.uint64))
    assert np.all(np.abs(g["echo_sums"] - o["echo_sums"]) <= RTOL * o["echo_sums"])


@pytest.mark.parametrize("bc", ["noflux", "periodic", "mirror"])
def test_voxel_division_with_labels_matches_oracle(bc):
    print(f"[test] divided labels bc={bc}", flush=True)
    dims = (16, 16, 16)
    solid, seeds, x, y, z, _ = _inputs(dims, 900, 12, 1)
    labels = R.voronoi_labels(solid, 9, 8, 4)
    delta = 1.0 - np.linspace(0.001, 0.02, 8)
    with R.Context(0) as ctx:
        img = R.Image.from_solid(ctx, solid, labels=labels, n_labels=8)
        g = R.cpmg_run(ctx, img, x, y, z, seeds, echoes=19, steps_per_echo=9, bc=bc, shift=1, label_delta=delta)
        img.close()
    o = O.walk(O.bitblock_pack(solid), dims, x, y, z, seeds, echoes=19, steps_per_echo=9, bc=bc, shift=1,
               labels=labels, label_delta=delta)
    _same(g, o)
    assert np.array_equal(g["energy"].view(np.uint64), o["energy"].view(np.uint64))
    assert np.all(np.abs(g["echo_sums"] - o["echo_sums"]) <= RTOL * o["echo_sums"])


def test_division_beyond_32_bit_addresses_takes_the_folded_walk():
    """A divided mirror image of more than 2^32 sub-voxel addresses."""
    print("[test] divided, folded fallback", flush=True)
    dims = (300, 20, 20)
    solid, seeds, x, y, z, pen = _inputs(dims, 200, 13, 8)
    with R.Context(0) as ctx:
        img = R.Image.from_solid(ctx, solid)
        g = R.cpmg_run(ctx, img, x, y, z, seeds, echoes=5, steps_per_echo=50, bc="mirror", shift=8, penalty=pen)
        img.close()
    o = O.walk(O.bitblock_pack(solid), dims, x, y, z, seeds, echoes=5, steps_per_echo=50, bc="mirror", shift=8,
               penalty=pen)
    _same(g, o)


def test_noalloc_run_that_narrow_blocks_would_split():
    """40,000 walkers and 4,000 echoes fit the static scratch with 256-thread
    blocks only; without an energy array the run has to stay one launch."""
    import ctypes as ct

    import torch

    from randomwalk_nmr_amd._lib import load
    from randomwalk_nmr_amd.core import _walker_struct, bc_code

    print("[test] noalloc, one launch", flush=True)
    n, echoes = 40_000, 4000
    solid, seeds, x, y, z, _ = _inputs((32, 32, 32), n, 8)
    L = load()
    out = []
    with R.Context(0) as ctx:
        img = R.Image.from_solid(ctx, solid)
        for fn in (L.rwnmr_cpmg_run, L.rwnmr_cpmg_run_noalloc):
            t = [torch.from_numpy(v.copy()).to("cuda") for v in (x, y, z, seeds.view(np.int64))]
            sums = torch.zeros(echoes + 1, dtype=torch.float64, device="cuda")
            w = _walker_struct(*t, None, None, None, 0.999, n, 1)
            torch.cuda.synchronize()
            code = fn(ctx.handle, img.handle, ct.byref(w), echoes, 1, bc_code("mirror"), 0,
                      ct.c_void_p(sums.data_ptr()))
            assert code == 0, L.rwnmr_last_error(ctx.handle)
            ctx.synchronize()
            out.append([v.cpu().numpy() for v in t] + [sums.cpu().numpy()])
        img.close()
    for a, b in zip(out[0][:4], out[1][:4]):
        assert np.array_equal(a, b)
    assert np.all(np.abs(out[0][4] - out[1][4]) <= RTOL * out[1][4])
