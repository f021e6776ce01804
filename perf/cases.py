"""Workloads of the mutual-interaction library, for timing and for comparing outputs.

Every case is one call (or the short sequence of calls) that a program built
on ncorpion_amd makes, on synthetic thin disks around a central body of mass 1
(G = 1; semi-major axes uniform in [0.9, 1.1], Rayleigh eccentricities 0.01 and
inclinations 0.005): the field, NcorpiON's brute-force and mesh integrators,
the RK4 driver, ensembles, the adjoint, and the calls a drop-in NcorpiON makes
on host arrays.
"""
import math

import numpy as np
import torch

from ncorpion_amd import Context, ic
from ncorpion_amd.autograd import RK4Trajectory

DT = 2.0 * math.pi / 256.0
_ctx = None


def context():
    """The program's one library context."""
    global _ctx
    if _ctx is None:
        _ctx = Context(0)
    return _ctx


# -- the cases -----------------------------------------------------------------

def listed():
    return [
        # What NcorpiON's own integrator calls every step through the drop-in,
        # at the size of its default brute-force runs: vector_field, then
        # brute_force, on host arrays (each call uploads its bodies).
        dict(name="dropin_2k", kind="dropin", n=2000, radius=2e-4),
        # The same run resident on the GPU: 64 steps of the brute-force
        # integrator with collisions in one call, in the reference's arithmetic.
        dict(name="leapfrog_exact_2k", kind="leapfrog", n=2000, precision="exact", steps=64,
             radius=2e-4, holes=0.0),
        # A larger brute-force run with the mixed field, collisions on.
        dict(name="leapfrog_mixed_64k", kind="leapfrog", n=65536, precision="mixed", steps=4,
             radius=2e-4, holes=0.0),
        # One field evaluation on device arrays in each precision: the exact
        # one at an odd size, the FP64 one with slots that bodies have left and
        # softening, the mixed one of the mutual terms alone.
        dict(name="field_exact_20k", kind="field", n=20011, precision="exact", softening=1e-3,
             holes=0.0, central=True),
        dict(name="field_fast64_50k", kind="field", n=50021, precision="fast64", softening=1e-3,
             holes=0.05, central=True),
        dict(name="field_mixed_100k", kind="field", n=100003, precision="mixed", softening=1e-6,
             holes=0.0, central=False),
        # One RK4 step of the 262,144-body disk of the benchmark.
        dict(name="rk4_mixed_262k", kind="rk4", n=262144, precision="mixed", softening=1e-6,
             steps=1, graph=False),
        # NcorpiON's mesh integrator: its ordinary size with the reference's
        # arithmetic, and a 2^20-body disk with the FP64 and the exact field.
        dict(name="mesh_exact_16k", kind="mesh", n=16384, precision="exact", steps=10, radius=1e-3),
        dict(name="mesh_fast64_1m", kind="mesh", n=1 << 20, precision="fast64", steps=4,
             radius=5e-5),
        dict(name="mesh_exact_1m", kind="mesh", n=1 << 20, precision="exact", steps=2,
             radius=5e-5),
        # 512 independent disks of 256 to 8192 bodies advanced together.
        dict(name="ensemble_512", kind="ensemble", systems=512, low=256, high=8192,
             precision="mixed", steps=2, radius=2e-4),
        # Training through a trajectory: forward with checkpoints, backward to
        # the initial state, the masses and the central body.
        dict(name="adjoint_16k", kind="adjoint", n=16384, steps=20, every=10, softening=1.0),
    ]


def _size(rng, lo, hi):
    """Log-uniform integer of [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["dropin", "leapfrog", "leapfrog", "field", "field", "field", "rk4", "mesh",
                       "mesh", "ensemble", "adjoint"])
    radius = rng.choice([1e-4, 2e-4])
    if kind == "dropin":
        return dict(kind=kind, n=_size(rng, 300, 8000), radius=radius)
    precision = rng.choice(["exact", "fast64", "mixed"])
    if kind == "leapfrog":
        n = _size(rng, 300, 12000 if precision == "exact" else 65536)
        steps = 64 if n <= 4000 else 16 if n <= 16384 else 4
        return dict(kind=kind, n=n, precision=precision, steps=steps, radius=radius,
                    holes=rng.choice([0.0, 0.1]))
    if kind == "field":
        top = {"exact": 32000, "fast64": 120000, "mixed": 262144}[precision]
        return dict(kind=kind, n=_size(rng, 500, top), precision=precision,
                    softening=rng.choice([0.0, 1e-6, 1e-3, 1.0]), holes=rng.choice([0.0, 0.05]),
                    central=rng.choice([True, False]))
    if kind == "rk4":
        precision = rng.choice(["fast64", "mixed"])
        n = _size(rng, 1000, 90000 if precision == "fast64" else 200000)
        return dict(kind=kind, n=n, precision=precision, softening=rng.choice([0.0, 1e-6]),
                    steps=8 if n <= 20000 else 1, graph=n <= 20000)
    if kind == "mesh":
        n = _size(rng, 8000, 1 << 20)
        return dict(kind=kind, n=n, precision=rng.choice(["exact", "fast64"]),
                    steps=4 if n <= 200000 else 2, radius=round(5e-5 * ((1 << 20) / n) ** 0.7, 7))
    if kind == "ensemble":
        low = rng.choice([64, 256])
        return dict(kind=kind, systems=_size(rng, 8, 512), low=low,
                    high=rng.choice([1024, 8192]), precision=rng.choice(["fast64", "mixed"]),
                    steps=rng.choice([1, 2]), radius=radius)
    return dict(kind=kind, n=_size(rng, 500, 12000), steps=rng.choice([5, 10, 20]),
                every=rng.choice([5, 10]), softening=1.0)


# -- inputs --------------------------------------------------------------------

def _disk(n, gen, mass, radius):
    """(n, 8) bodies on the device (the recipe of ncorpion_amd.ic.disk)."""
    dev = "cuda"

    def uni(lo, hi):
        return lo + (hi - lo) * torch.rand(n, generator=gen, dtype=torch.float64, device=dev)

    def rayleigh(sigma):
        u = torch.rand(n, generator=gen, dtype=torch.float64, device=dev)
        return sigma * torch.sqrt(-2.0 * torch.log1p(-u))

    a, e, inc = uni(0.9, 1.1), rayleigh(0.01).clamp(max=0.9), rayleigh(0.005)
    mean, om, node = (uni(0.0, 2.0 * math.pi) for _ in range(3))
    ecc = mean + e * torch.sin(mean)
    for _ in range(12):
        ecc = ecc - (ecc - e * torch.sin(ecc) - mean) / (1.0 - e * torch.cos(ecc))
    ce, se = torch.cos(ecc), torch.sin(ecc)
    b = a * torch.sqrt(1.0 - e * e)
    px, py, r = a * (ce - e), b * se, a * (1.0 - e * ce)
    rate = a ** -1.5
    vx, vy = -a * rate * se * a / r, b * rate * ce * a / r
    co, so, cn, sn = torch.cos(om), torch.sin(om), torch.cos(node), torch.sin(node)
    ci, si = torch.cos(inc), torch.sin(inc)
    rot = ((cn * co - sn * so * ci, -cn * so - sn * co * ci),
           (sn * co + cn * so * ci, -sn * so + cn * co * ci),
           (so * si, co * si))
    out = torch.empty((n, 8), dtype=torch.float64, device=dev)
    for k, (p, q) in enumerate(rot):
        out[:, k] = p * px + q * py
        out[:, 3 + k] = p * vx + q * vy
    out[:, 6] = mass
    out[:, 7] = radius
    return out


def _log_masses(n, gen):
    """Masses log-uniform in [1e-11, 1e-9] and radii 1e-4 (m / 1e-10)^(1/3)."""
    u = torch.rand(n, generator=gen, dtype=torch.float64, device="cuda")
    m = 1e-11 * torch.exp(u * math.log(100.0))
    return m, 1e-4 * (m / 1e-10) ** (1.0 / 3.0)


def _exists(n, gen, holes):
    if holes <= 0.0:
        return None
    return (torch.rand(n, generator=gen, device="cuda") >= holes).to(torch.int32)


def _central(count=None):
    c = torch.zeros((count or 1, 8), dtype=torch.float64, device="cuda")
    c[:, 6] = 1.0
    c[:, 7] = 1.0
    return c if count else c[0].contiguous()


def _sizes(case):
    return ic.seeded_ensemble_sizes(case["systems"], case["low"], case["high"])


def _mesh_params(n):
    # Cells of 0.01 where the disk is dense, else about 100 neighbours a body.
    return dict(gam=max(0.01, math.sqrt(14.0 / n)), gam_min=0.01, how_many_neighbours=100.0,
                disruption_threshold=0.05, high_dumping_threshold=100.0, cells=256)


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    s = dict(case=case, ctx=context())
    kind = case["kind"]
    if kind == "dropin":
        s["bodies"] = _disk(case["n"], gen, 1e-8, case["radius"]).cpu().numpy()
        s["central"] = (0.0, 0.0, 0.0, 1.0)
    elif kind in ("leapfrog", "mesh"):
        mass = 1e-8 if kind == "leapfrog" else 1e-10
        s["start"] = _disk(case["n"], gen, mass, case["radius"])
        s["exists"] = _exists(case["n"], gen, case.get("holes", 0.0))
        s["bodies"] = torch.empty_like(s["start"])
        s["central0"], s["central"] = _central(), _central()
    elif kind == "field":
        m, r = _log_masses(case["n"], gen)
        s["bodies"] = _disk(case["n"], gen, m, r)
        s["exists"] = _exists(case["n"], gen, case["holes"])
        s["central"] = (0.0, 0.0, 0.0, 1.0) if case["central"] else None
        s["acc"] = torch.zeros((case["n"], 3), dtype=torch.float64, device="cuda")
        s["cm"] = torch.zeros(3, dtype=torch.float64, device="cuda") if case["central"] else None
    elif kind == "rk4":
        m, r = _log_masses(case["n"], gen)
        s["start"] = _disk(case["n"], gen, m, r)
        s["bodies"] = torch.empty_like(s["start"])
        s["central0"], s["central"] = _central(), _central()
    elif kind == "ensemble":
        sizes = _sizes(case)
        s["offsets"] = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
        s["start"] = _disk(int(sizes.sum()), gen, 1e-8, case["radius"])
        s["bodies"] = torch.empty_like(s["start"])
        s["central0"], s["central"] = _central(case["systems"]), _central(case["systems"])
    else:
        b = _disk(case["n"], gen, 1e-8, 2e-4)
        s["x"], s["v"], s["m"] = (t.clone().requires_grad_(True)
                                  for t in (b[:, 0:3], b[:, 3:6], b[:, 6]))
        s["radius"] = b[:, 7].clone()
        s["central"] = _central().requires_grad_(True)
        s["target"] = b[:, 0:3] + 1e-3 * torch.randn((case["n"], 3), generator=gen,
                                                     dtype=torch.float64, device="cuda")
    return s


# -- one pass ------------------------------------------------------------------

def run(s):
    case, ctx = s["case"], s["ctx"]
    kind = case["kind"]
    if kind == "dropin":
        acc, cm = ctx.gravity_allpairs(s["bodies"], None, s["central"], 1.0, 0.0, "exact")
        b = s["bodies"].copy()
        ops = ctx.builtin_ops(b, DT, f=1.5)
        hits = ctx.brute_force_pass(b, None, DT, ops=ops)
        return acc, cm, b, hits
    if kind == "field":
        ctx.gravity_allpairs_dev(s["bodies"], s["acc"], s["exists"], s["central"], 1.0,
                                 case["softening"], case["precision"], s["cm"])
        return s["acc"], s["cm"]
    if kind == "adjoint":
        leaves = (s["x"], s["v"], s["m"], s["central"])
        for t in leaves:
            t.grad = None
        xt, vt, ct = RK4Trajectory.apply(s["x"], s["v"], s["m"], s["radius"], s["central"], 1.0,
                                         case["softening"], DT, case["steps"], case["every"], ctx)
        loss = (xt - s["target"]).square().sum() / case["n"]
        loss.backward()
        return [xt, vt, ct, loss] + [t.grad for t in leaves]
    # The integrators advance the program's arrays in place: each pass starts
    # from the same state.
    s["bodies"].copy_(s["start"])
    s["central"].copy_(s["central0"])
    if kind == "leapfrog":
        hits = ctx.leapfrog_dev(s["bodies"], s["central"], case["steps"], DT, 1.0, 0.0,
                                case["precision"], 1.5, 0, s["exists"], graph=True,
                                half_drift_start=True)
        return s["bodies"], s["central"], hits
    if kind == "rk4":
        ctx.rk4_steps_dev(s["bodies"], s["central"], case["steps"], DT, 1.0, case["softening"],
                          case["precision"], graph=case["graph"])
        return s["bodies"], s["central"]
    if kind == "mesh":
        params = _mesh_params(case["n"])
        hits = ctx.mesh_leapfrog_dev(s["bodies"], s["central"], case["steps"], DT / 2, params, 1.0,
                                     0.0, case["precision"], 1.5, 0, half_kick_start=True)
        return s["bodies"], s["central"], hits, params["gam"]
    hits = ctx.ensemble_rk4_dev(s["bodies"], s["offsets"], s["central"], case["steps"], DT, 1.0,
                                0.0, case["precision"], graph=True, collisions=True,
                                collision_f=1.5)
    return s["bodies"], s["central"], hits


# -- what a pass cannot do without ----------------------------------------------

def work(case):
    """20 flop an ordered interaction, 27 a collision test of a pair, 40 an
    interaction of the vector-Jacobian product; each body's 64 bytes read and
    written once a pass."""
    kind = case["kind"]
    if kind == "ensemble":
        sizes = _sizes(case).astype(np.float64)
        pairs, n = float((sizes * (sizes - 1.0)).sum()), float(sizes.sum())
        return {"bytes": 128.0 * n, "flops": case["steps"] * pairs * (4 * 20.0 + 13.5)}
    n = case["n"]
    pairs = float(n) * (n - 1)
    if kind == "dropin":
        return {"bytes": 64.0 * n + 24.0 * n + 128.0 * n, "flops": pairs * (20.0 + 13.5)}
    if kind == "leapfrog":
        return {"bytes": 128.0 * n, "flops": case["steps"] * pairs * (20.0 + 13.5)}
    if kind == "field":
        return {"bytes": 88.0 * n, "flops": 20.0 * pairs * (1.0 - case["holes"]) ** 2}
    if kind == "rk4":
        return {"bytes": 128.0 * n, "flops": case["steps"] * 4 * 20.0 * pairs}
    if kind == "mesh":
        # Ordered neighbours: bodies of the 3 x 3 cells around, on a disk of
        # area pi (1.1^2 - 0.9^2).
        gam = _mesh_params(n)["gam"]
        near = float(n) * n * 9.0 * gam * gam / (math.pi * 0.4)
        return {"bytes": case["steps"] * 128.0 * n, "flops": case["steps"] * near * (20.0 + 13.5)}
    return {"bytes": 128.0 * n, "flops": case["steps"] * 4 * pairs * (2 * 20.0 + 40.0)}


# -- the same outputs in plain 64-bit arithmetic ----------------------------------

def _field64(x, m, reach, G=1.0):
    """Mutual accelerations; reach: softening length of each body."""
    out = torch.empty_like(x)
    n = x.shape[0]
    step = max(1, (1 << 27) // n)
    for lo in range(0, n, step):
        hi = min(n, lo + step)
        d = [x[None, :, k] - x[lo:hi, None, k] for k in range(3)]
        r2 = d[0] * d[0]
        r2.addcmul_(d[1], d[1]).addcmul_(d[2], d[2])
        if float(reach.max()) > 0.0:
            r2 += (reach[None, :] + reach[lo:hi, None]).square_()
        i = torch.arange(lo, hi, device=x.device)
        r2[i - lo, i] = 1.0
        w = r2.rsqrt()
        w = w * w * w * (G * m)[None, :]
        w[i - lo, i] = 0.0
        for k in range(3):
            out[lo:hi, k] = (w * d[k]).sum(1)
    return out


def exact(case, seed):
    """The field cases by direct summation; the integrators' outputs are held
    to what the arithmetic they promise gives."""
    if case["kind"] != "field":
        return None
    s = prepare(case, seed)
    b = s["bodies"]
    on = torch.ones(case["n"], dtype=torch.bool, device="cuda")
    if s["exists"] is not None:
        on = s["exists"] != 0
    x, m, r = b[on, 0:3].contiguous(), b[on, 6].contiguous(), b[on, 7].contiguous()
    a = _field64(x, m, case["softening"] * r)
    cm = None
    if s["central"] is not None:
        t = x / x.square().sum(1, keepdim=True) ** 1.5
        a = a - t
        cm = (m[:, None] * t).sum(0)
    acc = torch.zeros((case["n"], 3), dtype=torch.float64, device="cuda")
    acc[on] = a
    return acc, cm
