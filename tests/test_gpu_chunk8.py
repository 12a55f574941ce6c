"""The 8-byte chunk cache (form 6) on noflux, periodic and mirror images, the
address displacements of images of periods of 128 and more, and the sizes at
which an unconfigured context sorts the walkers or changes its block: bit-exact
walkers against the oracle or the forms asked for by name, echo sums to 1e-12."""
import numpy as np
import pytest

import oracle as O
import randomwalk_nmr_amd as R

pytestmark = pytest.mark.gpu

RTOL = 1e-12


def _inputs(dims, n, seed):
    W, H, D = dims
    rng = np.random.default_rng(seed)
    solid = (rng.random((D, H, W)) < 0.3).astype(np.uint8)
    w = R.setup_walkers(solid, seed, n)
    return solid, w["seed"], w["x"], w["y"], w["z"], 1.0 - rng.uniform(0.001, 0.02, n)


@pytest.mark.parametrize("bc", ["noflux", "periodic", "mirror"])
@pytest.mark.parametrize("dims", [(2, 2, 2), (13, 9, 21), (64, 64, 64), (128, 160, 130), (127, 128, 256)])
@pytest.mark.parametrize("form", [3, 6])
def test_forms_match_oracle(bc, dims, form):
    print(f"[test] form={form} bc={bc} dims={dims}", flush=True)
    solid, seeds, x, y, z, pen = _inputs(dims, 801, 4)
    with R.Context(0) as ctx:
        ctx.set_unfolded(form)
        img = R.Image.from_solid(ctx, solid)
        g = R.cpmg_run(ctx, img, x, y, z, seeds, echoes=6, steps_per_echo=257, bc=bc, penalty=pen)
        m = R.map_run(ctx, img, x, y, z, seeds, steps=6 * 257, bc=bc)
        img.close()
    o = O.walk(O.bitblock_pack(solid), dims, x, y, z, seeds, echoes=6, steps_per_echo=257, bc=bc, penalty=pen)
    for k in ("x", "y", "z", "seed", "hits"):
        assert np.array_equal(g[k], o[k]), k
        assert np.array_equal(m[k], o[k]), k
    assert np.array_equal(g["energy"].view(np.uint64), o["energy"].view(np.uint64))
    assert np.all(np.abs(g["echo_sums"] - o["echo_sums"]) <= RTOL * o["echo_sums"])


@pytest.mark.parametrize("bc,n,steps", [("mirror", 65_537, 20), ("mirror", 70_001, 10_400), ("noflux", 400_001, 8),
                                        ("periodic", 400_001, 8), ("mirror", 524_287, 60), ("mirror", 524_288, 60),
                                        ("mirror", 70_001, 9_996), ("periodic", 70_001, 10_000),
                                        ("mirror", 524_287, 5_000), ("mirror", 524_288, 5_000),
                                        ("mirror", 600_001, 4_400)])
def test_unconfigured_runs_match_named_forms(bc, n, steps):
    """Default choices against form 3, unsorted: above the speculative walk, both
    sides of the line from which runs are sorted (10,000 steps of up to 250,000
    walkers, 2 ms of more), and sorted runs below, at and above the 1024-thread
    blocks of 524,288 walkers, with tiles of whole blocks and balanced ones.
    The unsorted lines of larger images follow below."""
    print(f"[test] default choice bc={bc} n={n} steps={steps}", flush=True)
    # balanced tiles need periods of 128 and more
    solid, seeds, x, y, z, pen = _inputs((72, 64, 64) if n > 600_000 else (40, 32, 24), n, 9)
    out = []
    for asked in (False, True):
        with R.Context(0) as ctx:
            if asked:
                ctx.set_unfolded(3)
                ctx.set_launch(256, 1)
                ctx.set_locality(False)
            img = R.Image.from_solid(ctx, solid)
            out.append(R.cpmg_run(ctx, img, x, y, z, seeds, echoes=4, steps_per_echo=steps // 4, bc=bc, penalty=pen))
            img.close()
    for k in ("x", "y", "z", "seed", "hits", "energy"):
        assert np.array_equal(out[0][k], out[1][k]), k
    assert np.all(np.abs(out[0]["echo_sums"] - out[1]["echo_sums"]) <= RTOL * out[1]["echo_sums"])


@pytest.mark.parametrize("dims,n", [((64, 64, 64), 262_145), ((96, 96, 96), 500_000), ((96, 96, 96), 500_001),
                                    ((127, 128, 128), 250_001), ((127, 128, 128), 400_001),
                                    ((128, 128, 128), 200_001), ((128, 128, 128), 300_001),
                                    ((128, 160, 130), 327_680), ((128, 160, 130), 327_681)])
@pytest.mark.parametrize("bc", ["periodic", "mirror"])
def test_unsorted_lines_match_the_plain_form(dims, n, bc):
    """Image sizes and walker counts at which an unsorted run changes its chunk,
    and a CPMG run its way to resolve a wall, against the unfolded walk without
    a chunk cache: one more flush than the shortest interval, odd step counts."""
    print(f"[test] unsorted lines bc={bc} dims={dims} n={n}", flush=True)
    solid, seeds, x, y, z, pen = _inputs(dims, n, 9)
    out = []
    for asked in (False, True):
        with R.Context(0) as ctx:
            if asked:
                ctx.set_unfolded(1)
                ctx.set_launch(256, 1)
                ctx.set_locality(False)
            img = R.Image.from_solid(ctx, solid)
            out.append(R.cpmg_run(ctx, img, x, y, z, seeds, echoes=3, steps_per_echo=43, bc=bc, penalty=pen))
            m = R.map_run(ctx, img, x, y, z, seeds, steps=129, bc=bc)
            img.close()
        for k in ("x", "y", "z", "seed", "hits"):
            assert np.array_equal(m[k], out[-1][k]), k
    for k in ("x", "y", "z", "seed", "hits", "energy"):
        assert np.array_equal(out[0][k], out[1][k]), k
    assert np.all(np.abs(out[0]["echo_sums"] - out[1]["echo_sums"]) <= RTOL * out[1]["echo_sums"])
