"""The work that a user of this framework has it do, as cases that can be timed.

A case is a dict of plain values; ``kind`` says which public call it makes:

* ``force``    - ``ForceContext.compute_forces_device``: the integrator's force call (particle mesh + tree walk);
* ``pm``       - the same call with the tree switched off (``TreePMForce.new_pm_only``'s use);
* ``step``     - ``ForceContext.step_device``: one leapfrog step, in the reference's drift-kick-drift order or
                 kick-drift-kick, launched eagerly or replayed as a captured graph;
* ``ensemble`` - ``Ensemble.compute_forces_device``: a parameter scan of uneven boxes in one call;
* ``poisson``  - ``PoissonSolver``'s mesh solve on device grids.

Particle sets follow the two recipes of ``janus_treepm.synth`` (a lattice with Zel'dovich displacements, m- on the
offset lattice with the negated field; NFW halos and uniform m+ with m- in the voids), drawn on the GPU so that new
inputs are quick to make.  Masses are m+ = 1 and |m-| = 19 as in the benchmark workloads.
"""
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "janus-sim_amd"))

import janus_treepm as jtp  # noqa: E402

M_PLUS, M_MINUS = 1.0, 19.0
PAIR_FLOPS = 38  # of one softened pair force with the split factor


def listed():
    return [
        # the smallest box in use (the smoke test's): launches and latency count
        dict(name="force_f32_20k", kind="force", recipe="halos", n=20_000, box=100.0, n_cells=32, precision="f32", leaf=4),
        # the small lattice configuration of the benchmark, in both precisions
        dict(name="force_f32_lattice_524k", kind="force", recipe="lattice", n=2 * 64 ** 3, box=250.0, n_cells=64,
             precision="f32", leaf=8),
        dict(name="force_f64_lattice_524k", kind="force", recipe="lattice", n=2 * 64 ** 3, box=250.0, n_cells=64,
             precision="f64", leaf=8),
        # the YAML fields alone (no split scale given): r_cut of 2 cells, r_s = r_cut / 3, theta 0.7; odd particle count
        dict(name="force_f32_yaml_1000003", kind="force", recipe="halos", n=1_000_003, box=120.0, n_cells=128,
             precision="f32", leaf=4, config=True),
        # an eighth of the headline box in the FP64 form (energy checks, reference runs)
        dict(name="force_f64_halos_2750k", kind="force", recipe="halos", n=2_750_000, box=125.0, n_cells=128,
             precision="f64", leaf=4),
        # the headline box
        dict(name="force_f32_halos_22M", kind="force", recipe="halos", n=22_000_000, box=250.0, n_cells=256,
             precision="f32", leaf=4),
        # the long-range part alone, at the headline size
        dict(name="pm_f32_halos_22M", kind="pm", recipe="halos", n=22_000_000, box=250.0, n_cells=256, precision="f32",
             leaf=4),
        # the reference's step (drift, kick with Hubble friction, drift) on initial-condition-like particles
        dict(name="step_dkd_f32_4M", kind="step", recipe="lattice", n=2 * 128 ** 3, box=500.0, n_cells=128,
             precision="f32", leaf=4, scheme="dkd", graph=False),
        # the large production box: kick-drift-kick, replayed as a graph
        dict(name="step_kdk_graph_f32_41M", kind="step", recipe="halos", n=2 * 256 ** 3 + 7_200_000, box=300.0,
             n_cells=512, precision="f32", leaf=4, scheme="kdk", graph=True),
        # a parameter scan: 16 boxes of 2 x 32^3 to 2 x 128^3 particles
        dict(name="ensemble_f32_16", kind="ensemble", boxes=16, lo=32, hi=128, precision="f32"),
        # the mesh solver by itself: the headline mesh, and the FP64 default on a smaller one
        dict(name="poisson_f32_256", kind="poisson", n_cells=256, box=250.0, precision="f32", r_s=1.25, deconvolve=1,
             k_min=0),
        dict(name="poisson_f64_128", kind="poisson", n_cells=128, box=200.0, precision="f64", r_s=0.0, deconvolve=0,
             k_min=2),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mesh_for(n, rng):
    """A power-of-two mesh of about one cell per particle, or half as fine."""
    g = 2 ** int(round(math.log2(n) / 3.0 - rng.choice((0.0, 0.35))))
    return min(512, max(32, g))  # r_cut of 5.6 cells may not exceed a fifth of the box


def draw(rng):
    kind = rng.choice(("force", "force", "force", "force", "pm", "step", "step", "ensemble", "poisson"))
    if kind == "poisson":
        prec = rng.choice(("f32", "f64"))
        return dict(kind=kind, n_cells=rng.choice((16, 32, 64, 128, 256, 512)), box=round(rng.uniform(50.0, 500.0), 2),
                    precision=prec, r_s=rng.choice((0.0, 1.25, 0.8)), deconvolve=rng.randrange(2), k_min=rng.choice((0, 2)))
    if kind == "ensemble":
        lo = rng.randint(24, 48)
        return dict(kind=kind, boxes=rng.randint(3, 24), lo=lo, hi=rng.randint(lo + 8, 112), precision="f32")
    prec = rng.choice(("f32", "f32", "f64")) if kind != "step" else "f32"
    recipe = rng.choice(("lattice", "halos"))
    hi = {"f32": 20_000_000, "f64": 2_500_000}[prec]
    n = _log_int(rng, 8_000, hi)
    if recipe == "lattice":
        n = 2 * max(16, int(round((n / 2) ** (1.0 / 3.0)))) ** 3
    else:
        n |= 1
    case = dict(kind=kind, recipe=recipe, n=n, box=round(rng.uniform(50.0, 400.0), 2), n_cells=_mesh_for(n, rng),
                precision=prec, leaf=rng.choice((4, 4, 8, 1, 13)))
    if kind == "force":
        case["theta"] = rng.choice((0.5, 0.5, 0.4, 0.7))
        case["group"] = rng.choice((32, 32, 32, 16, 64))
        case["split"] = rng.choice(("gauss", "gauss", "gauss", "erfc", "poly4"))
    if kind == "step":
        case["scheme"] = rng.choice(("dkd", "kdk"))
        case["graph"] = rng.random() < 0.5
    return case


# ------------------------------------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _fixed(x, box):
    """Positions (any period) to 32-bit fixed point, held in int32."""
    t = x / box + 0.5
    t = t - torch.floor(t)
    u = (t * 4294967296.0).to(torch.int64) & 0xFFFFFFFF
    return torch.where(u >= 2 ** 31, u - 2 ** 32, u).to(torch.int32).contiguous()


def _lattice(n_side, box, g):
    """n_side^3 m+ displaced by random long waves (rms 0.3 spacings, power ~ k^-2.5), m- on the offset lattice with the
    negated displacement."""
    h = box / n_side
    c = (torch.arange(n_side, device="cuda", dtype=torch.float64) + 0.5) * h - box / 2
    q = torch.stack(torch.meshgrid(c, c, c, indexing="ij"), -1).reshape(-1, 3)
    waves = 24
    k = torch.randint(-4, 5, (waves, 3), device="cuda", generator=g).to(torch.float64)
    k[:, 0] = torch.where(k.abs().sum(1) == 0, torch.ones_like(k[:, 0]), k[:, 0])
    kn = k.norm(dim=1, keepdim=True)
    amp = torch.randn((waves, 1), device="cuda", generator=g, dtype=torch.float64) * kn ** -1.25
    phase = torch.rand((waves,), device="cuda", generator=g, dtype=torch.float64) * (2 * math.pi)
    psi = torch.zeros_like(q)
    for w in range(waves):
        psi += torch.sin(q @ k[w] * (2 * math.pi / box) + phase[w])[:, None] * (amp[w] * k[w] / kn[w])
    psi *= 0.3 * h / psi.square().sum(1).mean().sqrt()
    pos = torch.cat([q + psi, q + 0.5 * h - psi])
    sp = torch.ones(2 * len(q), dtype=torch.int8, device="cuda")
    sp[len(q):] = -1
    return pos, sp


def _halos(n, box, g):
    """Half m+ (60 % of them in NFW halos with a power-law mass function, the rest uniform), half m- in the cells where
    m+ is below its median."""
    n_plus = n // 2
    n_minus = n - n_plus
    n_in = int(0.6 * n_plus)
    halos = max(12, n // 11_000)
    f8 = dict(device="cuda", dtype=torch.float64)
    e, lo, hi = -0.9, 1e-5, 1e-2
    mass = (lo ** e + torch.rand(halos, generator=g, **f8) * (hi ** e - lo ** e)) ** (1.0 / e)
    cdf = torch.cumsum(mass, 0) / mass.sum()
    ids = torch.searchsorted(cdf, torch.rand(n_in, generator=g, **f8)).clamp_(max=halos - 1)
    counts = torch.bincount(ids, minlength=halos).to(torch.float64)
    conc = 5.0 + 10.0 * torch.rand(halos, generator=g, **f8)
    centre = (torch.rand((halos, 3), generator=g, **f8) - 0.5) * box
    r200 = (3.0 * counts / (800.0 * math.pi * n_plus / box ** 3)) ** (1.0 / 3.0)
    # radius / r200 by bisection of the enclosed NFW mass
    u, c = torch.rand(n_in, generator=g, **f8), conc[ids]
    target = u * (torch.log1p(c) - c / (1 + c))
    a, b = torch.zeros_like(u), torch.ones_like(u)
    for _ in range(24):
        m = 0.5 * (a + b)
        low = torch.log1p(c * m) - c * m / (1 + c * m) < target
        a, b = torch.where(low, m, a), torch.where(low, b, m)
    v = torch.randn((n_in, 3), generator=g, **f8)
    v /= v.norm(dim=1, keepdim=True)
    pos = [centre[ids] + (r200[ids] * 0.5 * (a + b))[:, None] * v,
           (torch.rand((n_plus - n_in, 3), generator=g, **f8) - 0.5) * box]
    plus = torch.cat(pos)
    # voids: coarse cells of about 64 particles
    m = max(4, int(round((n / 64) ** (1.0 / 3.0))))

    def cell(x):
        i = (torch.floor((x / box + 0.5) * m).to(torch.int64)) % m
        return (i[:, 2] * m + i[:, 1]) * m + i[:, 0]

    count = torch.bincount(cell(plus), minlength=m ** 3)
    void = count <= count.to(torch.float32).median()
    got, have = [], 0
    while have < n_minus:
        cand = (torch.rand((int((n_minus - have) * 2.2) + 1024, 3), generator=g, **f8) - 0.5) * box
        cand = cand[void[cell(cand)]][: n_minus - have]
        got.append(cand)
        have += len(cand)
    sp = torch.ones(n, dtype=torch.int8, device="cuda")
    sp[n_plus:] = -1
    return torch.cat([plus] + got), sp


def _particles(case, seed):
    g = _gen(seed)
    if case["recipe"] == "lattice":
        pos, sp = _lattice(int(round((case["n"] / 2) ** (1.0 / 3.0))), case["box"], g)
    else:
        pos, sp = _halos(case["n"], case["box"], g)
    order = torch.randperm(len(sp), generator=g, device="cuda")  # a simulation's particles are in no order
    return _fixed(pos[order], case["box"]), sp[order].contiguous()


def _params(case):
    prec = jtp.FP64 if case["precision"] == "f64" else jtp.FP32
    if case.get("config"):
        p = jtp.params_from_config(case["box"], case["n_cells"], n_particles=case["n"])
    else:
        p = jtp.default_params(case["box"], case["n_cells"])
        p.softening = case["box"] / case["n"] ** (1.0 / 3.0) / 30.0
    p.precision = prec
    p.leaf_size = case["leaf"]
    if "theta" in case:
        p.theta = case["theta"]
        p.theta_cut = 0.66 * case["theta"]
    if "group" in case:
        p.group_size = case["group"]
    p.split_mode = {"gauss": jtp.SPLIT_ERFC_GAUSS, "erfc": jtp.SPLIT_ERFC, "poly4": jtp.SPLIT_POLY4}[case.get("split", "gauss")]
    if case["kind"] == "pm":
        p.tree_enabled = 0
    return p


def _real(case):
    return torch.float64 if case["precision"] == "f64" else torch.float32


def _ensemble_boxes(case):
    """The scan's box list, the same for every seed: lattice sides log-uniform between lo and hi."""
    rng = random.Random(1000 + case["boxes"])
    out = []
    for _ in range(case["boxes"]):
        side = _log_int(rng, case["lo"], case["hi"])
        cells = 2 ** int(round(math.log2(2 * side ** 3) / 3.0))
        out.append(dict(kind="force", recipe="lattice", n=2 * side ** 3, box=rng.uniform(100.0, 500.0),
                        n_cells=min(256, max(32, cells)), precision=case["precision"], leaf=4,
                        m_minus=rng.uniform(5.0, 40.0)))
    return out


def prepare(case, seed):
    kind = case["kind"]
    if kind == "poisson":
        # mass per cell of a smooth overdensity plus noise
        G = case["n_cells"]
        g = _gen(seed)
        rho = torch.randn((G, G, G), device="cuda", generator=g, dtype=torch.float64)
        rho = (1.0 + 0.5 * rho).to(_real(case)).contiguous()
        solver = jtp.PoissonSolver(G, case["box"], r_s=case["r_s"] * case["box"] / G, k_min=case["k_min"],
                                   precision=jtp.FP64 if case["precision"] == "f64" else jtp.FP32,
                                   deconvolve=case["deconvolve"])
        phi = torch.empty_like(rho)
        return dict(kind=kind, solver=solver, rho=_Grid(rho), phi=_Grid(phi))
    if kind == "ensemble":
        boxes = _ensemble_boxes(case)
        ens = jtp.Ensemble([_params(b) for b in boxes], [M_PLUS] * len(boxes), [b["m_minus"] for b in boxes])
        parts = [_particles(b, 1000 * seed + i) for i, b in enumerate(boxes)]
        acc = [torch.empty((b["n"], 3), device="cuda", dtype=_real(case)) for b in boxes]
        torch.cuda.synchronize()
        return dict(kind=kind, ens=ens, n=[b["n"] for b in boxes], parts=parts, acc=acc)
    pos, sp = _particles(case, seed)
    n = len(sp)
    ctx = jtp.ForceContext(_params(case), M_PLUS, M_MINUS)
    acc = torch.zeros((n, 3), device="cuda", dtype=_real(case))
    state = dict(kind=kind, ctx=ctx, n=n, pos=pos, sp=sp, acc=acc)
    torch.cuda.synchronize()
    if kind == "step":
        # a step starts from the forces of the step before, at velocities that those have built up over some steps
        ctx.compute_forces_device(n, pos.data_ptr(), sp.data_ptr(), acc.data_ptr())
        h = case["box"] / case["n_cells"]
        rms = float(acc.double().square().mean().sqrt())
        state["dt"] = 0.02 * math.sqrt(h / rms)  # the typical particle gains ~ 4e-4 cells of displacement a step
        state["vel"] = (acc * (5.0 * state["dt"])).contiguous()
        state["scheme"] = jtp.STEP_KDK if case["scheme"] == "kdk" else jtp.STEP_DKD
        state["graph"] = case["graph"]
        state["hubble"] = 0.01 / state["dt"]
        state["scale"] = case["box"] / 4294967296.0
        torch.cuda.synchronize()
    return state


class _Grid:
    """A torch grid where the solver takes a device array (it reads the pointer)."""

    def __init__(self, t):
        self.t, self.ptr = t, t.data_ptr()


def run(state):
    kind = state["kind"]
    if kind in ("force", "pm"):
        state["ctx"].compute_forces_device(state["n"], state["pos"].data_ptr(), state["sp"].data_ptr(),
                                           state["acc"].data_ptr())
        return state["acc"]
    if kind == "step":
        state["ctx"].step_device(state["n"], state["pos"].data_ptr(), state["vel"].data_ptr(), state["sp"].data_ptr(),
                                 state["acc"].data_ptr(), state["dt"], hubble_plus=state["hubble"],
                                 scheme=state["scheme"], graph=state["graph"])
        # positions as a program shows or stores them: lengths in [-L/2, L/2), float32
        x = torch.bitwise_xor(state["pos"], -2 ** 31).to(torch.float32).mul_(state["scale"])
        return {"x": x, "v": state["vel"], "a": state["acc"]}
    if kind == "ensemble":
        state["ens"].compute_forces_device(state["n"], [p.data_ptr() for p, _ in state["parts"]],
                                           [s.data_ptr() for _, s in state["parts"]],
                                           [a.data_ptr() for a in state["acc"]])
        return state["acc"]
    state["solver"].ctx.pm_solve_device(state["rho"], state["phi"])
    return state["phi"].t


# ------------------------------------------------------------------------------------------------ work and exact
def _pairs(case, p):
    """Pair forces a particle cannot do without: the sources within r_cut at the mean density, at most the ~1200 terms
    that an opening angle of 0.5 leaves of a clustered neighbourhood."""
    return min(1200.0, case["n"] * 4.0 / 3.0 * math.pi * p.r_cut ** 3 / p.box_size ** 3)


def _fft_work(G, real):
    """One mesh solve: the grid in, the potential out, a real transform each way and the Green product."""
    cells = float(G) ** 3
    return dict(bytes=2 * cells * real, flops=2 * 2.5 * cells * math.log2(cells) + 3 * cells)


def work(case):
    kind = case["kind"]
    real = 8 if case["precision"] == "f64" else 4
    if kind == "poisson":
        return _fft_work(case["n_cells"], real)
    if kind == "ensemble":
        each = [work(b) for b in _ensemble_boxes(case)]
        return dict(bytes=sum(w["bytes"] for w in each), flops=sum(w["flops"] for w in each))
    n, p = case["n"], _params(case)
    w = dict(bytes=n * (13 + 3 * real), flops=n * 250.0)  # position and species in, force out; weights and gradient
    solve = _fft_work(case["n_cells"], real)
    w["bytes"] += 2 * solve["bytes"]  # two interlaced meshes
    w["flops"] += 2 * solve["flops"]
    if kind != "pm":
        w["flops"] += n * _pairs(case, p) * PAIR_FLOPS
    if kind == "step":
        w["bytes"] += n * (2 * 3 * real + 12 + 12)  # velocity in and out, position out, position as lengths out
    return w


def _axis(G, **kw):
    i = torch.arange(G, **kw)
    return torch.where(i > G // 2, i - G, i)


def _solve64(rho, box, r_s, k_min, deconvolve, matched):
    """Potential of the mass grid rho [z][y][x] in 64 bits: -4 pi G / k^2 exp(-k^2 r_s^2), optionally over the squared
    CIC window (twice: deposit and interpolation) and times the match to the 4-point gradient stencil."""
    G = rho.shape[0]
    dev = rho.device
    h = box / G
    ki = _axis(G, device=dev, dtype=torch.float64)
    k1 = ki * (2 * math.pi / box)
    KZ, KY, KX = k1[:, None, None], k1[None, :, None], k1[None, None, : G // 2 + 1].abs()
    k2 = KX ** 2 + KY ** 2 + KZ ** 2
    keep = torch.maximum(torch.maximum(ki.abs()[:, None, None], ki.abs()[None, :, None]),
                         ki.abs()[None, None, : G // 2 + 1]) >= max(k_min, 1)
    k2s = torch.where(k2 > 0, k2, torch.ones_like(k2))
    green = -4 * math.pi / k2s * torch.exp(-k2 * r_s ** 2) / h ** 3
    if deconvolve:
        def win(k):
            x = 0.5 * k * h
            return torch.where(x.abs() > 0, torch.sin(x) / torch.where(x.abs() > 0, x, torch.ones_like(x)), torch.ones_like(x)) ** 2

        green = green / (win(KX) * win(KY) * win(KZ)) ** 2
    if matched:
        def stencil(k):
            return (8 * torch.sin(k * h) - torch.sin(2 * k * h)) / (6 * h)

        DX, DY, DZ = stencil(KX), stencil(KY), stencil(KZ)
        kd = KX * DX + KY * DY + KZ * DZ
        d2 = DX ** 2 + DY ** 2 + DZ ** 2
        green = green * kd / torch.maximum(d2, 0.25 * k2s)
    spec = torch.fft.rfftn(rho) * torch.where(keep, green, torch.zeros_like(green))
    return torch.fft.irfftn(spec, s=(G, G, G))


def _pm64(case, seed):
    """Long-range accelerations of a pm case in 64 bits: CIC on two meshes half a cell apart, the solve, the 4-point
    gradient and CIC back, averaged over the two."""
    pos, sp = _particles(case, seed)
    G, box = case["n_cells"], case["box"]
    p = _params(case)
    u = (pos.to(torch.int64) & 0xFFFFFFFF).to(torch.float64) * (G / 4294967296.0)
    del pos
    q = torch.where(sp > 0, M_PLUS, -M_MINUS).to(torch.float64)
    out = torch.zeros((len(sp), 3), device="cuda", dtype=torch.float64)
    for shift in (0.0, 0.5):
        x = u + shift
        i0 = torch.floor(x)
        f = x - i0
        i0 = i0.to(torch.int64)
        rho = torch.zeros(G ** 3, device="cuda", dtype=torch.float64)

        def corners():
            for c in range(8):
                d = (c & 1, c >> 1 & 1, c >> 2)
                w = torch.ones_like(q)
                idx = torch.zeros_like(i0[:, 0])
                for a in (2, 1, 0):
                    w = w * (f[:, a] if d[a] else 1 - f[:, a])
                    idx = idx * G + (i0[:, a] + d[a]) % G
                yield w, idx

        for w, idx in corners():
            rho.index_add_(0, idx, w * q)
        phi = _solve64(rho.reshape(G, G, G), box, p.r_s, p.k_min, True, True)
        h = box / G
        for a, dim in enumerate((2, 1, 0)):
            r = lambda s: torch.roll(phi, -s, dim)  # noqa: E731
            grad = ((8 * (r(1) - r(-1)) - (r(2) - r(-2))) / (12 * h)).reshape(-1)
            acc = torch.zeros_like(q)
            for w, idx in corners():
                acc += w * grad[idx]
            out[:, a] -= 0.5 * acc * torch.sign(q)
    return out


def _ewald64(case, seed):
    """Accelerations of all particles in the periodic box in 64 bits: the real-space sum over nearest images (softened,
    split at L / 14) and the reciprocal sum over |k_i| <= 10."""
    pos, sp = _particles(case, seed)
    p = _params(case)
    L, eps2, n = case["box"], p.softening ** 2, len(sp)
    x = (pos.to(torch.int64) & 0xFFFFFFFF).to(torch.float64) / 4294967296.0 * L
    q = torch.where(sp > 0, M_PLUS, -M_MINUS).to(torch.float64)
    r_s = L / 14.0 / 2.0
    acc = torch.zeros_like(x)
    step = max(1, 32_000_000 // n)
    for s in range(0, n, step):
        d = x[None, :, :] - x[s:s + step, None, :]
        d -= L * torch.round(d / L)
        r2 = d.square().sum(-1) + eps2
        r = r2.sqrt()
        t = r / (2 * r_s)
        w = q[None, :] * (torch.erfc(t) + 2 / math.sqrt(math.pi) * t * torch.exp(-t * t)) / (r2 * r)
        acc[s:s + step] = (w[:, :, None] * d).sum(1)
    m = 10
    for i in range(0, m + 1):
        for j in range(-m, m + 1):
            for k in range(-m, m + 1):
                if (i, j, k) <= (0, 0, 0):
                    continue
                kv = torch.tensor([i, j, k], device="cuda", dtype=torch.float64) * (2 * math.pi / L)
                k2 = float(kv.square().sum())
                ph = x @ kv
                c, s = torch.cos(ph), torch.sin(ph)
                amp = 2 * 4 * math.pi / (k2 * L ** 3) * math.exp(-k2 * r_s ** 2)
                acc += (amp * (c * (q * s).sum() - s * (q * c).sum()))[:, None] * kv
    return acc * torch.sign(q)[:, None]


def exact(case, seed):
    kind = case["kind"]
    if kind == "poisson":
        G = case["n_cells"]
        rho = torch.randn((G, G, G), device="cuda", generator=_gen(seed), dtype=torch.float64)
        rho = (1.0 + 0.5 * rho).to(_real(case)).double()
        return _solve64(rho, case["box"], case["r_s"] * case["box"] / G, case["k_min"], case["deconvolve"],
                        case["deconvolve"])
    if kind == "pm":
        return _pm64(case, seed)
    # the periodic force itself is within reach for the smallest boxes; the tree's own approximation is the error there
    if kind == "force" and case["n"] <= 30_000 and case.get("split", "gauss") == "gauss":
        return _ewald64(case, seed)
    return None
