"""The measured workloads of the framework: what a user has it do, through
its public entry points, from the smallest host call to the full-size runs.

listed() names the workloads, draw() gives others of the same ranges;
prepare() makes what a program has in hand before the call (image, walkers,
context, model), run() is one pass, work() what a pass cannot do without, and
exact() the same result from a plain 64-bit torch walker.

Images are sphere packs and walkers are placed in the pore space by the
framework's own generators, as its benchmark and tests do.  Where walkers
are device tensors a pass starts by copying their start state, since the
calls update them in place."""
import math
import random

import numpy as np
import torch

import randomwalk_nmr_amd as R
from randomwalk_nmr_amd.fit import CpmgModel

DEV = "cuda:0"
D0 = 2.5                 # um^2 / ms
N_LABELS = 8
GYRO = 42.576            # MHz / T
# 32-bit operations that a walker-step cannot do without: three 64-bit
# shift-xors (12), the residue, the move and the wall test
STEP_OPS = 16

KINDS = ("cpmg", "divided", "map", "pfgse", "gradient", "jacobian", "population", "batch", "field")


def listed():
    return [
        # the headline benchmark: 512^3, 1M walkers, 10,000 echoes of 12 steps on mirror
        # boundaries, in the 1024-thread blocks its autotuner settles on
        dict(name="cpmg-512-1M", kind="cpmg", W=512, H=512, D=512, r0=6.0, r1=16.0, phi=0.20, n=1_000_000,
             echoes=10_000, spe=12, bc="mirror", voxel=0.5, rho=25.0, host=False, hits=False, spread=False,
             threads=1024),
        # the benchmark's small run: few walkers, latency counts
        dict(name="cpmg-128-10k", kind="cpmg", W=128, H=128, D=128, r0=8.0, r1=8.0, phi=0.25, n=10_000, echoes=2000,
             spe=3, bc="mirror", voxel=1.0, rho=10.0, host=False, hits=False, spread=False, threads=0),
        # the smallest call: numpy arrays in and out, a few hundred steps (the smoke test)
        dict(name="cpmg-32-host", kind="cpmg", W=32, H=32, D=32, r0=4.0, r1=4.0, phi=0.3, n=2000, echoes=50, spe=3,
             bc="mirror", voxel=1.0, rho=10.0, host=True, hits=True, spread=False, threads=0),
        # the reference's default boundary on an image of odd sides, a relaxivity per walker,
        # hits counted
        dict(name="cpmg-noflux-odd", kind="cpmg", W=211, H=150, D=97, r0=4.0, r1=10.0, phi=0.30, n=200_000,
             echoes=500, spe=4, bc="noflux", voxel=1.0, rho=15.0, host=False, hits=True, spread=True, threads=0),
        # voxel division (each voxel walked as 2 x 2 x 2), host arrays as the command line has them
        dict(name="cpmg-divided", kind="divided", W=100, H=100, D=100, r0=4.0, r1=8.0, phi=0.30, n=50_000, echoes=200,
             spe=8, bc="mirror", voxel=1.0, rho=10.0, shift=1),
        # hit counts for the collision histograms, periodic image of odd sides
        dict(name="map-periodic-odd", kind="map", W=160, H=130, D=95, r0=5.0, r1=9.0, phi=0.35, n=300_000, steps=2000,
             bc="periodic"),
        # the PFGSE benchmark: 16 diffusion times x 64 gradients x 2 relaxivities
        dict(name="pfgse-256-1M", kind="pfgse", W=256, H=256, D=256, r0=10.0, r1=10.0, phi=0.30, n=1_000_000,
             n_delta=16, n_k=64, t0=0.5, t1=40.0, sets=2, bc="mirror", host=False, even=True),
        # a small PFGSE from host arrays: the reference's fixed list of unevenly spaced gradients,
        # noflux, a relaxivity per walker
        dict(name="pfgse-host-noflux", kind="pfgse", W=101, H=90, D=83, r0=5.0, r1=8.0, phi=0.35, n=30_000, n_delta=6,
             n_k=33, t0=0.5, t1=20.0, sets=0, bc="noflux", host=True, even=False),
        # one evaluation of the gradient fit: decay forward, then the backward replay
        dict(name="fit-gradient", kind="gradient", W=256, H=256, D=256, r0=6.0, r1=12.0, phi=0.25, n=1_000_000,
             echoes=2000, spe=3, bc="mirror"),
        # one evaluation of the least-squares fit: decay and its Jacobian
        dict(name="fit-jacobian", kind="jacobian", W=160, H=160, D=160, r0=6.0, r1=12.0, phi=0.25, n=250_000,
             echoes=1000, spe=3, bc="mirror"),
        # uneven instances in one launch
        dict(name="batch-uneven", kind="batch", count=16, side0=64, side1=192, n0=10_000, n1=250_000, echoes=1000,
             spe=3, bc="mirror"),
        # CPMG in an internal field
        dict(name="field-odd", kind="field", W=150, H=120, D=101, r0=5.0, r1=9.0, phi=0.30, n=100_000, echoes=200,
             spe=8, bc="periodic"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _dims(rng, lo, hi):
    """Sides over [lo, hi]: a cube of a power of two, or three sides of their own."""
    if rng.random() < 0.35:
        s = 1 << rng.randint(math.ceil(math.log2(lo)), int(math.log2(hi)))
        return dict(W=s, H=s, D=s)
    return {k: _log(rng, lo, hi) for k in ("W", "H", "D")}


def _pack(rng):
    r0 = round(rng.uniform(3.0, 8.0), 2)
    return dict(r0=r0, r1=round(r0 + rng.uniform(0.0, 6.0), 2), phi=round(rng.uniform(0.15, 0.40), 3))


def draw(rng):
    """One more case of the ranges above; the fit also scores a population of
    the genetic algorithm on one trajectory."""
    kind = rng.choice(("cpmg", "cpmg", "cpmg") + KINDS[1:])
    bc = rng.choice(("mirror", "mirror", "periodic", "noflux"))
    if kind == "cpmg":
        host = rng.random() < 0.3
        n = _log(rng, 1000, 100_000 if host else 1_000_000)
        spe = rng.randint(1, 16)
        echoes = max(20, min(_log(rng, 50, 4000), int(2e10 / (n * spe))))
        return dict(kind=kind, **_dims(rng, 24, 256), **_pack(rng), n=n, echoes=echoes, spe=spe, bc=bc, voxel=1.0,
                    rho=round(rng.uniform(5.0, 40.0), 2), host=host, hits=rng.random() < 0.5,
                    spread=rng.random() < 0.4, threads=rng.choice((0, 0, 1024)))
    if kind == "divided":
        shift = rng.randint(1, 2)
        return dict(kind=kind, **_dims(rng, 24, 128), **_pack(rng), n=_log(rng, 1000, 100_000),
                    echoes=_log(rng, 20, 300), spe=rng.randint(4, 12), bc=bc, voxel=1.0,
                    rho=round(rng.uniform(5.0, 40.0), 2), shift=shift)
    if kind == "map":
        return dict(kind=kind, **_dims(rng, 24, 256), **_pack(rng), n=_log(rng, 2000, 1_000_000),
                    steps=_log(rng, 200, 5000), bc=bc)
    if kind == "pfgse":
        host = rng.random() < 0.5
        return dict(kind=kind, **_dims(rng, 40, 192), **_pack(rng), n=_log(rng, 2000, 100_000 if host else 1_000_000),
                    n_delta=rng.randint(2, 16), n_k=rng.randint(8, 80), t0=0.5, t1=round(rng.uniform(5.0, 40.0), 2),
                    sets=rng.choice((0, 1, 2, 4)), bc=bc, host=host, even=rng.random() < 0.6)
    if kind in ("gradient", "jacobian", "population"):
        return dict(kind=kind, **_dims(rng, 32, 192), **_pack(rng), n=_log(rng, 5000, 500_000),
                    echoes=_log(rng, 100, 1500), spe=rng.randint(1, 8), bc=bc)
    if kind == "batch":
        return dict(kind=kind, count=rng.randint(3, 16), side0=rng.randint(24, 64), side1=rng.randint(70, 160),
                    n0=_log(rng, 1000, 10_000), n1=_log(rng, 20_000, 150_000), echoes=_log(rng, 100, 1000),
                    spe=rng.randint(2, 6), bc=bc)
    return dict(kind=kind, **_dims(rng, 24, 160), **_pack(rng), n=_log(rng, 2000, 200_000),
                echoes=_log(rng, 20, 300), spe=2 * rng.randint(1, 6), bc=bc)


# ------------------------------------------------------------------ inputs

def _solid(c, seed):
    """Solid voxels [D, H, W]; images of 512 a side are eight mirrored packs
    of half the side."""
    W, H, D = c["W"], c["H"], c["D"]
    if W >= 512:
        half, _ = R.sphere_pack(W // 2, H // 2, D // 2, c["r0"], c["r1"], c["phi"], seed)
        for ax in range(3):
            half = np.concatenate([half, np.flip(half, ax)], ax)
        return np.ascontiguousarray(half)
    return R.sphere_pack(W, H, D, c["r0"], c["r1"], c["phi"], seed)[0]


def _penalties(c, n, seed):
    """(per-walker deltas or None, uniform delta)"""
    d = R.penalty(c.get("rho", 10.0), c.get("voxel", 1.0), D0)
    if not c.get("spread"):
        return None, d
    return 1.0 - (1.0 - d) * np.random.default_rng(seed).uniform(0.2, 1.8, n), d


def _dev(a):
    a = np.ascontiguousarray(a)
    return torch.from_numpy(a.view(np.int64) if a.dtype == np.uint64 else a).to(DEV)


def _walkers(solid, c, seed):
    """x, y, z, seed of n walkers in the pore space."""
    if c.get("shift"):
        w = R.setup_walkers(solid, seed, c["n"], shift=c["shift"])
        return [w[k] for k in ("x", "y", "z", "seed")]
    seeds, x, y, z = R.seed_and_place(solid, seed, c["n"])
    return [x, y, z, seeds]


def _pfgse_inputs(c, seed):
    """(steps between diffusion times, wave vectors [n_k] or [n_delta, n_k], set deltas or None)"""
    dt = R.time_step(1.0, D0)
    deltas = np.geomspace(c["t0"], c["t1"], c["n_delta"])
    steps = np.array([int(round(d / dt)) for d in deltas])
    inc = np.diff(np.concatenate([[0], steps])).astype(np.uint32)
    if c["even"]:
        kx = np.linspace(0.0, 1.0, c["n_k"])[None, :] * (3.0 / np.sqrt(D0 * deltas))[:, None]
    else:
        kx = np.sqrt(np.linspace(0.0, 1.0, c["n_k"])) * 3.0 / math.sqrt(D0 * c["t0"])
    k = [kx, np.zeros_like(kx), np.zeros_like(kx)]
    sets = None
    if c["sets"]:
        sets = np.array([R.penalty(10.0 * q, 1.0, D0) for q in range(c["sets"])])
    return inc, k, sets


def _field(c, solid, seed):
    f = np.random.default_rng(seed).normal(0.0, 1e-3, solid.shape)
    f[solid != 0] = 0.0
    return f


def _fit_inputs(c, seed):
    """(rho[8], T2b, target decay) of a fit evaluation; a population has 16 rows."""
    rng = np.random.default_rng(seed)
    rho = rng.uniform(5.0, 40.0, (16, N_LABELS) if c["kind"] == "population" else N_LABELS)
    t2b = rng.uniform(2000.0, 3500.0, 16) if c["kind"] == "population" else 2800.0
    t = np.arange(c["echoes"] + 1) * c["spe"] * R.time_step(1.0, D0)
    return rho, t2b, np.exp(-t / 150.0) + rng.normal(0.0, 0.005, c["echoes"] + 1)


def _sizes(c):
    """(side, walkers) of every instance of a batch: sides in 16s, walkers
    over a logarithmic range, in an order of their own."""
    rng = random.Random(c["count"] * 1000 + c["side1"])
    return [(rng.randint(c["side0"] // 16, c["side1"] // 16) * 16, _log(rng, c["n0"], c["n1"]))
            for _ in range(c["count"])]


def _instances(c, seed):
    """(solid, walkers, delta) of every instance of a batch."""
    rng = random.Random(seed)
    out = []
    for i, (side, n) in enumerate(_sizes(c)):
        r = rng.uniform(4.0, 10.0)
        solid, _ = R.sphere_pack(side, side, side, r, r, rng.uniform(0.15, 0.40), seed + i)
        out.append((solid, _walkers(solid, dict(n=n), seed + 100 + i), R.penalty(rng.uniform(5.0, 50.0), 1.0, D0)))
    return out


def prepare(case, seed):
    c = case
    ctx = R.Context(0)
    s = dict(c=c, ctx=ctx)
    if c["kind"] == "batch":
        made = _instances(c, seed)
        s["start"] = [_dev(np.concatenate([w[k] for _, w, _ in made])) for k in range(4)]
        s["walk"] = [t.clone() for t in s["start"]]
        s["energy"] = torch.ones(len(s["start"][0]), dtype=torch.float64, device=DEV)
        s["sums"] = torch.zeros((len(made), c["echoes"] + 1), dtype=torch.float64, device=DEV)
        s["inst"], at = [], 0
        for i, (solid, w, delta) in enumerate(made):
            m = slice(at, at + len(w[0]))
            at = m.stop
            x, y, z, sd = (t[m] for t in s["walk"])
            s["inst"].append(dict(img=R.Image.from_solid(ctx, solid), x=x, y=y, z=z, seed=sd, energy=s["energy"][m],
                                  echo_sums=s["sums"][i], echoes=c["echoes"], steps_per_echo=c["spe"], bc=c["bc"],
                                  delta=delta))
        return s
    solid = _solid(c, seed)
    w = _walkers(solid, c, seed + 1)
    if c["kind"] in ("gradient", "jacobian", "population"):
        img = R.Image.from_solid(ctx, solid, R.voronoi_labels(solid, 64, N_LABELS, seed + 2), N_LABELS)
        s["model"] = CpmgModel(ctx, img, *w, echoes=c["echoes"], steps_per_echo=c["spe"], voxel=1.0, D0=D0, bc=c["bc"])
        s["rho"], s["t2b"], target = _fit_inputs(c, seed)
        s["target"] = torch.from_numpy(target)
        return s
    s["img"] = R.Image.from_solid(ctx, solid)
    if c.get("threads"):
        ctx.set_launch(c["threads"], 1)
    pen, s["delta"] = _penalties(c, c["n"], seed + 3)
    f64 = dict(dtype=torch.float64, device=DEV)
    if c["kind"] == "divided" or c.get("host"):
        s["start"], s["pen"] = w, pen
        if c["kind"] == "pfgse":
            s["inc"], s["k"], s["sets"] = _pfgse_inputs(c, seed)
        return s
    s["start"] = [_dev(a) for a in w]
    s["walk"] = [t.clone() for t in s["start"]]
    s["pen"] = None if pen is None else _dev(pen)
    s["hits"] = torch.zeros(c["n"], dtype=torch.int32, device=DEV) if c.get("hits") or c["kind"] == "map" else None
    if c["kind"] == "cpmg":
        s["energy"], s["sums"] = torch.ones(c["n"], **f64), torch.zeros(c["echoes"] + 1, **f64)
    if c["kind"] == "field":
        s["field"] = _dev(_field(c, solid, seed + 4))
        s["alive"], s["phase"] = torch.ones(c["n"], **f64), torch.zeros(c["n"], **f64)
        s["sums"] = torch.zeros(c["echoes"] + 1, **f64)
    if c["kind"] == "pfgse":
        inc, k, sets = _pfgse_inputs(c, seed)
        s["inc"], s["k"] = _dev(inc.view(np.int32)), [_dev(a) for a in k]
        s["sets"] = None if sets is None else _dev(sets)
        s["M"] = torch.zeros((max(c["sets"], 1), c["n_delta"], c["n_k"]), **f64)
        s["msd"] = torch.zeros((c["n_delta"], 3), **f64)
    return s


# -------------------------------------------------------------------- pass

def _reset(s):
    for a, b in zip(s["walk"], s["start"]):
        a.copy_(b)
    return s["walk"]


def run(s):
    c, ctx = s["c"], s["ctx"]
    kind = c["kind"]
    if kind in ("cpmg", "divided"):
        kw = dict(echoes=c["echoes"], steps_per_echo=c["spe"], bc=c["bc"], penalty=s["pen"], delta=s["delta"])
        if kind == "divided":
            return R.cpmg_run(ctx, s["img"], *s["start"], shift=c["shift"], **kw)
        if c["host"]:
            return R.cpmg_run(ctx, s["img"], *s["start"], **kw)
        x, y, z, sd = _reset(s)
        s["energy"].fill_(1.0)
        if s["hits"] is not None:
            s["hits"].zero_()
        return R.cpmg_run(ctx, s["img"], x, y, z, sd, energy=s["energy"], hits=s["hits"], echo_sums=s["sums"], **kw)
    if kind == "map":
        x, y, z, sd = _reset(s)
        s["hits"].zero_()
        return R.map_run(ctx, s["img"], x, y, z, sd, steps=c["steps"], bc=c["bc"], hits=s["hits"])
    if kind == "pfgse":
        kw = dict(steps_inc=s["inc"], kx=s["k"][0], ky=s["k"][1], kz=s["k"][2], voxel=1.0, bc=c["bc"],
                  penalty=s["pen"], delta=s["delta"], set_delta=s["sets"])
        if c["host"]:
            return R.pfgse_run(ctx, s["img"], *s["start"], **kw)
        x, y, z, sd = _reset(s)
        return R.pfgse_run(ctx, s["img"], x, y, z, sd, x0=s["start"][0], y0=s["start"][1], z0=s["start"][2],
                           M=s["M"], msd=s["msd"], **kw)
    if kind == "gradient":
        rho = torch.tensor(s["rho"], dtype=torch.float64, requires_grad=True)
        t2b = torch.tensor(s["t2b"], dtype=torch.float64, requires_grad=True)
        decay = s["model"].decay(rho, t2b).cpu()
        torch.mean((decay - s["target"]) ** 2).backward()
        return dict(decay=decay.detach(), rho=rho.grad, t2b=t2b.grad)
    if kind == "jacobian":
        decay, jac = s["model"].decay_and_jacobian(s["rho"], s["t2b"])
        return dict(decay=decay, jac=jac)
    if kind == "population":
        return dict(decay=s["model"].decays(s["rho"], s["t2b"]))
    if kind == "batch":
        x, y, z, sd = _reset(s)
        s["energy"].fill_(1.0)
        R.cpmg_batch_run(ctx, s["inst"])
        return dict(x=x, y=y, z=z, seed=sd, energy=s["energy"], echo_sums=s["sums"])
    x, y, z, sd = _reset(s)
    s["alive"].fill_(1.0)
    s["phase"].zero_()
    return R.cpmg_field_run(ctx, s["img"], x, y, z, sd, echoes=c["echoes"], steps_per_echo=c["spe"],
                            field=s["field"], gyromagnetic_ratio=GYRO, time_interval_ms=R.time_step(1.0, D0),
                            bc=c["bc"], delta=s["delta"], p_alive=s["alive"], phase=s["phase"], echo_sums=s["sums"])


# -------------------------------------------------------------------- work

def work(case):
    """Bytes: walker state in and out (positions 12, seed 8, energy or phase
    8 or 16), image bits (and labels, field), results; operations: STEP_OPS a
    walker-step, one multiply-add per PFGSE term."""
    c = case
    if c["kind"] == "batch":
        n, vox = sum(m for _, m in _sizes(c)), sum(side ** 3 for side, _ in _sizes(c))
        return {"bytes": 2 * 28 * n + vox / 8 + 8.0 * c["count"] * c["echoes"],
                "flops": float(STEP_OPS) * n * c["echoes"] * c["spe"]}
    n, vox = c["n"], c["W"] * c["H"] * c["D"]
    b, ops = 2 * 28.0 * n + vox / 8, 0.0
    if c["kind"] == "pfgse":
        steps = int(round(c["t1"] / R.time_step(1.0, D0)))
        ops = 2.0 * n * c["n_delta"] * c["n_k"] * max(c["sets"], 1)
    elif c["kind"] == "map":
        steps = c["steps"]
    else:
        steps = c["echoes"] * c["spe"]
        b += 8.0 * (c["echoes"] + 1)
    if c["kind"] in ("gradient", "jacobian", "population"):
        b += vox
    if c["kind"] == "gradient":
        steps *= 2
    if c["kind"] == "field":
        b += 8.0 * vox + 2 * 16.0 * n
    return {"bytes": b, "flops": ops + float(STEP_OPS) * n * steps}


# ------------------------------------------------------- 64-bit plain walker

class _Walk:
    """Walkers on a [D, H, W] solid volume, one step at a time, in plain
    torch: xorshift64, direction = state mod 6 (y-, x-, y+, x+, z+, z-), the
    boundary, then a move or a wall hit."""

    def __init__(self, solid, walkers, bc, shift=0):
        self.bc, self.shift = bc, shift
        self.dims = torch.tensor(solid.shape[::-1], device=DEV)
        self.solid = torch.from_numpy(solid.reshape(-1) != 0).to(DEV)
        self.pos = torch.stack([_dev(a).long() for a in walkers[:3]])
        self.s = _dev(walkers[3])
        axis = torch.tensor([1, 0, 1, 0, 2, 2], device=DEV)
        sign = torch.tensor([-1, -1, 1, 1, 1, -1], device=DEV)
        self.unit = torch.zeros((3, 6), dtype=torch.long, device=DEV)
        self.unit[axis, torch.arange(6, device=DEV)] = sign

    def voxel(self, pos):
        """Index of the image voxel that positions fall in."""
        d = self.dims[:, None]
        g = pos >> self.shift
        if self.bc == "periodic":
            g = g % d
        elif self.bc == "mirror":
            g = g % (2 * d)
            g = torch.minimum(g, 2 * d - 1 - g)
        return g[0] + self.dims[0] * (g[1] + self.dims[1] * g[2])

    def step(self):
        """Advance; returns (hit, voxel tried)."""
        s = self.s
        s = s ^ (s << 13)
        s = s ^ ((s >> 7) & ((1 << 57) - 1))
        self.s = s = s ^ (s << 17)
        u = self.unit[:, (((s >> 32) & 0xFFFFFFFF) * 4 + (s & 0xFFFFFFFF)) % 6]
        if self.bc == "noflux":
            g, d = self.pos >> self.shift, self.dims[:, None]
            u = torch.where(((u < 0) & (g == 0)) | ((u > 0) & (g == d - 1)), -u, u)
        new = self.pos + u
        at = self.voxel(new)
        hit = self.solid[at]
        self.pos = torch.where(hit, self.pos, new)
        return hit, at


def _cpmg(solid, w, delta, echoes, spe, bc, shift=0):
    walk = _Walk(solid, w, bc, shift)
    e = torch.ones(len(w[0]), dtype=torch.float64, device=DEV)
    sums = [e.sum()]
    for _ in range(echoes):
        for _ in range(spe):
            hit, _ = walk.step()
            e = torch.where(hit, e * delta, e)
        sums.append(e.sum())
    return e, torch.stack(sums)


def _labelled(c, solid, labels, w, delta):
    """Echo sums and the Jacobian by the log deltas."""
    walk = _Walk(solid, w, c["bc"])
    lab = torch.from_numpy(labels.reshape(-1)).to(DEV).long()
    e = torch.ones(c["n"], dtype=torch.float64, device=DEV)
    h = torch.zeros((c["n"], N_LABELS), dtype=torch.float64, device=DEV)
    sums, jac = [e.sum()], [h.T @ e]
    for _ in range(c["echoes"]):
        for _ in range(c["spe"]):
            hit, at = walk.step()
            t = lab[at]
            e = torch.where(hit, e * delta[t], e)
            h.scatter_add_(1, t[:, None], hit[:, None].double())
        sums.append(e.sum())
        jac.append((h * e[:, None]).sum(0))
    return torch.stack(sums), torch.stack(jac, 1)


def _steps_of(c):
    if c["kind"] == "map":
        return c["steps"]
    if c["kind"] == "pfgse":
        return int(round(c["t1"] / R.time_step(1.0, D0)))
    return c["echoes"] * c["spe"]


def exact(case, seed):
    c = case
    if c["kind"] == "map":
        return None       # whole numbers only
    n = sum(m for _, m in _sizes(c)) if c["kind"] == "batch" else c["n"]
    per_step = 2.5e-4 * c.get("count", 1) + 1.5e-9 * n
    if _steps_of(c) * per_step > 18.0:
        return None
    none = dict(x=None, y=None, z=None, seed=None, hits=None)
    if c["kind"] == "batch":
        es, sums = zip(*(_cpmg(solid, w, d, c["echoes"], c["spe"], c["bc"]) for solid, w, d in _instances(c, seed)))
        return dict(none, energy=torch.cat(es), echo_sums=torch.stack(sums))
    solid = _solid(c, seed)
    w = _walkers(solid, c, seed + 1)
    pen, delta = _penalties(c, c["n"], seed + 3)
    if pen is not None:
        delta = _dev(pen)
    if c["kind"] in ("cpmg", "divided"):
        e, sums = _cpmg(solid, w, delta, c["echoes"], c["spe"], c["bc"], c.get("shift", 0))
        return dict(none, energy=e, echo_sums=sums)
    if c["kind"] == "field":
        walk = _Walk(solid, w, c["bc"])
        f = _dev(_field(c, solid, seed + 4)).reshape(-1)
        gt = 0.5 * (1.0e6 * GYRO) * (1.0e-3 * R.time_step(1.0, D0))
        alive = torch.ones(c["n"], dtype=torch.float64, device=DEV)
        phase = torch.zeros_like(alive)
        sums = [alive.sum()]
        for _ in range(c["echoes"]):
            for _ in range(2):
                phase = -phase
                for _ in range(c["spe"] // 2):
                    phase = phase + gt * f[walk.voxel(walk.pos)]
                    hit, _ = walk.step()
                    alive = torch.where(hit, alive * delta, alive)
                    phase = phase + gt * f[walk.voxel(walk.pos)]
            sums.append((alive * torch.cos(phase)).sum())
        return dict(none, p_alive=alive, phase=phase, energy=None, echo_sums=torch.stack(sums))
    if c["kind"] == "pfgse":
        inc, k, sets = _pfgse_inputs(c, seed)
        walk = _Walk(solid, w, c["bc"])
        start = walk.pos
        rows = [torch.as_tensor(d, dtype=torch.float64, device=DEV) for d in ([delta] if sets is None else sets)]
        es = [torch.ones(c["n"], dtype=torch.float64, device=DEV) for _ in rows]
        M, msd = [], []
        for i, steps in enumerate(inc):
            h = torch.zeros(c["n"], dtype=torch.float64, device=DEV)
            for _ in range(int(steps)):
                h += walk.step()[0]
            es = [e * torch.pow(d, h) for e, d in zip(es, rows)]
            r = (walk.pos - start).double()
            ki = torch.from_numpy(np.stack([a[i] if a.ndim == 2 else a for a in k])).to(DEV)
            M.append([torch.stack([(e * torch.cos(ki[:, j] @ r)).sum() for j in range(c["n_k"])]) for e in es])
            msd.append((r * r).sum(1))
        M = torch.stack([torch.stack([M[i][q] for i in range(len(inc))]) for q in range(len(rows))])
        return dict(none, M=M, msd=torch.stack(msd), energy=es[0] if c["host"] else None)
    labels = R.voronoi_labels(solid, 64, N_LABELS, seed + 2)
    rho, t2b, target = _fit_inputs(c, seed)
    t = torch.arange(c["echoes"] + 1, dtype=torch.float64, device=DEV) * (c["spe"] * R.time_step(1.0, D0))
    slope = -(2.0 / 3.0) / (D0 * 1e3)
    if c["kind"] == "population":
        if 16 * _steps_of(c) * (4e-4 + 2e-9 * n) > 15.0:
            return None
        decays = []
        for r, b in zip(rho, t2b):
            M, _ = _labelled(c, solid, labels, w, _dev(1.0 + slope * r))
            decays.append(torch.exp(-t / b) * M / M[0])
        return dict(decay=torch.stack(decays))
    if _steps_of(c) * (4e-4 + 2e-9 * n) > 15.0:
        return None
    d = _dev(1.0 + slope * rho)
    M, J = _labelled(c, solid, labels, w, d)
    bulk = torch.exp(-t / t2b)
    S = bulk * M / M[0]
    drho = J / d[:, None] * slope * (bulk / M[0])
    if c["kind"] == "jacobian":
        return dict(decay=S, jac=torch.cat([(drho * _dev(rho)[:, None]).T, (S * t / t2b)[:, None]], 1))
    g = 2.0 * (S - _dev(target)) / len(S)
    return dict(decay=S, rho=drho @ g, t2b=(g * S * t).sum() / t2b ** 2)
