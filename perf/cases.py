"""The workloads that this framework's speed is judged by.

Every case builds a seeded synthetic system (copies of the 22-atom chain on a
lattice, as the benchmark's workloads), uploads it as a user's program does and
runs one pass through a public entry point:

  step        a captured MD step of the engine, replayed (a dynamics run)
  batch       the same for many umbrella windows in one model
  loop        one step as separate calls, one wrapper per term (the shape of a
              driver that brings its own step loop)
  isspa       the IS-SPA solvent force alone (a program that adds it to the
              forces of its own MD code)
  nonbond     the all-pairs force alone
  components  the FP64 force components (analysis, validation)
  match       one force-matching evaluation: differentiable forces of a batch
              of frames, the loss and its gradients

`exact` computes the same values in 64 bits with plain torch.  The
Monte-Carlo points are FP32 values by definition (counter-based generator), and
the three discontinuous decisions -- inside a sphere or not, the periodic image,
an Andersen collision -- are taken on FP32 values, as the model defines them.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "isspa-force-cuda_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from isspa_amd import batch, synth  # noqa: E402
from isspa_amd.system import UmbrellaRestraint  # noqa: E402

SPACING = 16.0      # lattice spacing of the 19,998-atom benchmark workload, A
LARGEST = 19998.0 ** 2 * 20


def listed():
    return [
        # the shortest dynamics run: one chain, where a step is launches and latency
        {"name": "step_22", "kind": "step", "chains": 1, "n_mc": 10, "steps": 10, "periodic": False,
         "restraint": False},
        # the size of the one run whose timings the reference publishes: a 44-atom dimer under an umbrella
        # restraint, 100 points an atom
        {"name": "step_44_umbrella", "kind": "step", "chains": 2, "n_mc": 100, "steps": 10,
         "periodic": False, "restraint": True},
        # an ordinary run, 50 chains
        {"name": "step_1100", "kind": "step", "chains": 50, "n_mc": 20, "steps": 5, "periodic": False,
         "restraint": False},
        # a ragged size in between, in a box small enough for the minimum image
        {"name": "step_4510_periodic", "kind": "step", "chains": 205, "n_mc": 20, "steps": 1,
         "periodic": True, "restraint": False},
        # the largest run, the headline workload
        {"name": "step_19998", "kind": "step", "chains": 909, "n_mc": 20, "steps": 1, "periodic": False,
         "restraint": False},
        # an umbrella-sampling campaign: 64 windows of uneven size in one model
        {"name": "batch_64", "kind": "batch", "ljpairs": 32, "small": 24, "big": 8, "n_mc": 20,
         "steps": 5},
        # a driver that calls each term itself, 25 chains
        {"name": "loop_550", "kind": "loop", "chains": 25, "n_mc": 20, "periodic": False},
        # the solvent force with many points an atom (the shipped 44-atom deck's nMC)
        {"name": "isspa_44_nmc1000", "kind": "isspa", "chains": 2, "n_mc": 1000, "periodic": False},
        # the all-pairs force of a mid-size system, periodic
        {"name": "nonbond_2222", "kind": "nonbond", "chains": 101, "periodic": True},
        # FP64 components of an ordinary system
        {"name": "components_1100", "kind": "components", "chains": 50, "n_mc": 20, "periodic": False},
        # force matching on one frame, and on a batch of frames
        {"name": "match_1x550", "kind": "match", "frames": 1, "chains": 25, "n_mc": 20},
        {"name": "match_32x1100", "kind": "match", "frames": 32, "chains": 50, "n_mc": 20},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "batch", "loop", "isspa", "nonbond", "components", "match"])
    if kind == "batch":
        return {"kind": kind, "ljpairs": rng.randint(0, 48), "small": rng.randint(1, 48),
                "big": rng.randint(0, 16), "n_mc": rng.choice([10, 20, 33]), "steps": 5}
    if kind == "match":
        return {"kind": kind, "frames": _log_int(rng, 1, 32), "chains": _log_int(rng, 2, 50),
                "n_mc": rng.choice([5, 10, 17, 20])}
    if kind == "nonbond":
        return {"kind": kind, "chains": _log_int(rng, 1, 909), "periodic": rng.random() < 0.5}
    chains = _log_int(rng, 1, {"step": 800, "loop": 300, "isspa": 400, "components": 100}[kind])
    n = 22.0 * chains
    top = min(1000.0, 0.8 * LARGEST / (n * n), 6.0e5 / n)
    c = {"kind": kind, "chains": chains, "n_mc": max(1, _log_int(rng, 5, max(6.0, top)))}
    c["periodic"] = rng.random() < 0.4
    if kind == "step":
        work_ = n * n * c["n_mc"]
        c["steps"] = 10 if work_ < 5.0e6 else 5 if work_ < 3.0e8 else 1
        c["restraint"] = chains > 1 and rng.random() < 0.3
    return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _system(case, seed):
    """`chains` rotated copies of the chain on a lattice, in a box twice the
    lattice (the minimum image never fires) or just holding it (periodic)."""
    chains = case["chains"]
    grid = max(1, math.ceil(chains ** (1.0 / 3.0) - 1e-9))
    region = SPACING * grid
    lbox = max(region, 30.0) if case.get("periodic") else max(200.0, 2.5 * region)
    s = synth.make_lattice(chains, region, grid, lbox, seed=1000 + seed)
    s.n_mc = case.get("n_mc", 20)
    s.temperature_k, s.pnu, s.seed = 298.0, 0.01, 12345 + seed
    synth.maxwell_velocities(s, seed=2000 + seed)
    if case.get("restraint"):
        s.us = UmbrellaRestraint.from_groups([0, 4], [22, 26], s.true_mass, 20.0, 15.0)
    return s


def _windows(case, seed):
    ws = batch.umbrella_windows(case["ljpairs"], case["small"], case["big"], n_mc=case["n_mc"],
                                seed=12348 + 100 * seed)
    rng = np.random.default_rng(3000 + seed)
    for w in ws:  # every seed its own coordinates
        w.xyzq[:, :3] += rng.normal(scale=0.02, size=(w.n_atoms, 3)).astype(np.float32)
    return batch.merge_windows(ws)


def _frames(case, seed):
    """A batch of frames of one topology: lattice positions with thermal noise."""
    import dataclasses
    base = _system(case, 0)
    rng = np.random.default_rng(4000 + seed)
    ws = []
    for _ in range(case["frames"]):
        f = dataclasses.replace(base)
        f.xyzq = base.xyzq.copy()
        f.xyzq[:, :3] += rng.normal(scale=0.1, size=(base.n_atoms, 3)).astype(np.float32)
        ws.append(f)
    merged = batch.merge_windows(ws)
    return base, merged


def _match_inputs(case, seed):
    """(model system, parameters, theta, q per atom of every frame, target)."""
    from isspa_amd.diff import DiffParams
    base, merged = _frames(case, seed)
    prm = DiffParams.from_system(base)
    rng = np.random.default_rng(5000 + seed)
    theta = prm.theta * (1.0 + rng.uniform(-0.05, 0.05, prm.theta.shape))
    theta[:, 3] = np.maximum(theta[:, 3], 1.05)
    q = np.tile(prm.q + rng.uniform(-0.9, 0.9, prm.q.shape), case["frames"])
    target = rng.normal(scale=10.0, size=(merged.n_atoms, 3))
    return merged, prm, theta, q, target


def prepare(case, seed):
    kind = case["kind"]
    if kind == "match":
        from isspa_amd.diff import DiffForces
        system, prm, theta, q, target = _match_inputs(case, seed)
        dev = torch.device("cuda:0")
        t = lambda a: torch.as_tensor(a, dtype=torch.float64, device=dev)  # noqa: E731
        return {"kind": kind, "model": DiffForces(system, prm), "theta": t(theta).requires_grad_(),
                "q": t(q).requires_grad_(), "target": t(target),
                "norm": float((target ** 2).mean())}
    from isspa_amd.engine import GpuSystem
    system = _windows(case, seed) if kind == "batch" else _system(case, seed)
    g = GpuSystem(system, "cuda:0")
    if kind in ("step", "batch"):
        g.set_step(0)
        g.capture(case["steps"])
    return {"kind": kind, "gpu": g, "step": 0}


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    kind = state["kind"]
    if kind == "match":
        from isspa_amd.diff import isspa_forces
        theta, q = state["theta"], state["q"]
        theta.grad = q.grad = None
        f = isspa_forces(theta, q, state["model"])
        loss = ((f - state["target"]) ** 2).mean() / state["norm"]
        loss.backward()
        return {"forces": f, "loss": loss, "grad_theta": theta.grad, "grad_q": q.grad}
    g, step = state["gpu"], state["step"]
    state["step"] += 1
    if kind in ("step", "batch"):
        g.replay(1)
        return {"x": g.x, "v": g.v, "f": g.f}
    if kind == "components":
        return {**{"isspa_" + k: v for k, v in g.isspa_components(step).items()},
                **{"nonbond_" + k: v for k, v in g.nonbond_components().items()}}
    g.zero_forces()
    if kind == "isspa":
        return {"f": g.isspa_force(step)}
    if kind == "nonbond":
        return {"f": g.nonbond_force()}
    _, energies = g.bonded_force()
    g.isspa_force(step)
    g.nonbond_force()
    g.leapfrog(step)
    return {"x": g.x, "v": g.v, "f": g.f, "energies": energies}


def work(case):
    """Inputs read once and outputs written once; 24 FLOP per (point, atom) of
    the field pass, 70 of the force pass and 36 per unordered atom pair (the
    benchmark's counting); the adjoint at the forward's count."""
    kind = case["kind"]
    if kind == "batch":
        sizes = [2] * case["ljpairs"] + [22] * case["small"] + [220] * case["big"]
    else:
        sizes = [22 * case["chains"]] * case.get("frames", 1)
    n, nsq = float(sum(sizes)), float(sum(k * k for k in sizes))
    solvent = 94.0 * nsq * case.get("n_mc", 0)
    pairs = 18.0 * nsq
    if kind in ("step", "batch"):
        return {"bytes": case["steps"] * 80.0 * n, "flops": case["steps"] * (solvent + pairs)}
    if kind == "nonbond":
        return {"bytes": 32.0 * n, "flops": pairs}
    if kind == "isspa":
        return {"bytes": 32.0 * n, "flops": solvent}
    if kind == "match":
        return {"bytes": 100.0 * n, "flops": 2.0 * (solvent + pairs)}
    return {"bytes": (160.0 if kind == "components" else 80.0) * n, "flops": solvent + pairs}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
_DEV = "cuda" if torch.cuda.is_available() else "cpu"
_PAIRS = 40_000_000  # pairs of one piece of a pass


def _f32(a):
    return torch.as_tensor(np.asarray(a, np.float32), device=_DEV)


def _f64(a):
    return torch.as_tensor(np.asarray(a), device=_DEV, dtype=torch.float64)


def _i64(a):
    return torch.as_tensor(np.asarray(a), device=_DEV, dtype=torch.int64)


def _mulhilo(c, x):
    """High and low words of the 32 x 32 bit product, in int64 arithmetic."""
    lo16 = c * (x & 0xFFFF)
    mid = c * (x >> 16) + (lo16 >> 16)
    return mid >> 16, ((mid & 0xFFFF) << 16) | (lo16 & 0xFFFF)


def _philox(index, stream, draw_, step, sys_id, seed):
    """Philox4x32-10 (Salmon et al., SC'11): counter {index, stream | draw,
    step, system}, key = seed."""
    m = 0xFFFFFFFF
    c = [index, torch.full_like(index, (stream << 24) | draw_), torch.full_like(index, step & m),
         torch.full_like(index, sys_id & m)]
    k0, k1 = seed & m, (seed >> 32) & m
    for _ in range(10):
        h0, l0 = _mulhilo(0xD2511F53, c[0])
        h1, l1 = _mulhilo(0xCD9E8D57, c[2])
        c = [h1 ^ c[1] ^ k0, l1, h0 ^ c[3] ^ k1, l0]
        k0, k1 = (k0 + 0x9E3779B9) & m, (k1 + 0xBB67AE85) & m
    return c


def _points(x32, rmax, n_mc, seed, step, sys_id):
    """MC points of one window (FP32): the first draw on the 24-bit lattice
    inside the ball |u|^2 < 0.99, scaled by the owner's rmax."""
    n = x32.shape[0]
    idx = torch.arange(n * n_mc, device=_DEV, dtype=torch.int64)
    v = torch.zeros((n * n_mc, 3), dtype=torch.int64, device=_DEV)
    todo = torch.ones(n * n_mc, dtype=torch.bool, device=_DEV)
    for d in range(64):
        o = _philox(idx, 0, d, step, sys_id, seed)
        c = torch.stack([2 * (w >> 8) - (1 << 24) for w in o[:3]], dim=1)
        ok = todo & ((c * c).sum(1) <= 278660226943549)
        v[ok] = c[ok]
        todo &= ~ok
        if not bool(todo.any()):
            break
    u = v.to(torch.float32) * 2.0 ** -24
    own = torch.repeat_interleave(torch.arange(n, device=_DEV), n_mc)
    return x32[own] + rmax[own][:, None] * u, own


def _separations(a32, b32, box):
    """Pairs a x b: separations in 64 bits (the image decided on the FP32
    difference) and the FP32 squared distance of the sphere tests."""
    half = np.float32(0.5) * np.float32(box)
    r64, d2 = [], None
    for k in range(3):
        d = a32[:, None, k] - b32[None, :, k]
        img = (d > float(half)).to(torch.float64) - (d < -float(half)).to(torch.float64)
        r64.append(a32[:, None, k].double() - b32[None, :, k].double() - img * float(np.float32(box)))
        d = (d.double() - img * float(np.float32(box))).float().double()
        # one rounding an axis: a product and its fused sums
        d2 = (d * d).float().double() if d2 is None else (d * d + d2).float().double()
    return r64, d2


def _moments(x):
    """<P1>, <P2>, <P3> of the Langevin distribution."""
    h = 0.5 * x * x
    s, first = [], 1.0
    for l in range(4):
        first = first / (2 * l + 1) if l else 1.0
        t = torch.full_like(x, first)
        acc = t
        for k in range(40):
            t = t * h / ((k + 1) * (2 * l + 2 * k + 3))
            acc = acc + t
        s.append(acc)
    big = torch.clamp(x, min=4.0)
    c1 = 1.0 / torch.tanh(big) - 1.0 / big
    c2 = 1.0 - 3.0 * c1 / big
    c3 = c1 - 5.0 * c2 / big
    lo = x < 5.0
    return (torch.where(lo, x * s[1] / s[0], c1), torch.where(lo, x * x * s[2] / s[0], c2),
            torch.where(lo, x ** 3 * s[3] / s[0], c3))


def _constants():
    """The model's constants, evaluated in FP32 as the library's defaults."""
    f = np.float32
    ep, p0 = f(2.3473), f(4.173705894203977)
    e0 = f(3.0) / (f(4.0) * f(3.1415926535) * f(0.0075) * p0) * (f(1.0) - f(1.0) / ep)
    return {"e0": float(e0), "p0": float(p0), "q0": float(f(1.6899960102882601)),
            "o0": float(f(9.3658298730779350)), "ep": float(ep)}


class _Tables:
    """g, E (read at the g bin) and F of the IS-SPA tables, by linear interpolation."""

    def __init__(self, it):
        pad = lambda a: _f64(np.concatenate([a, np.zeros((a.shape[0], 1), a.dtype)], axis=1))  # noqa: E731
        self.g, self.e, self.f = pad(it.g), pad(it.e), pad(it.f)
        self.ng, self.nf = it.g.shape[1], it.f.shape[1]
        self.grids = [(float(r0), float(dr), float(np.float32(1.0) / np.float32(dr)))
                      for r0, dr in (it.g_grid, it.e_grid, it.f_grid)]

    def g_and_e(self, t, d):
        (g0, gd, gi), (e0, ed, ei) = self.grids[:2]
        b = torch.trunc((d - g0) * gi).long()
        c = b.clamp(0, self.ng - 2)
        ph, phe = (d - (g0 + c * gd)) * gi, (d - (e0 + c * ed)) * ei
        g = self.g[t, c + 1] * ph + self.g[t, c] * (1.0 - ph)
        e = self.e[t, c + 1] * phe + self.e[t, c] * (1.0 - phe)
        mid = (b >= 0) & (b < self.ng - 1)
        g = torch.where(mid, g, (b >= 0).to(g.dtype))
        return g, torch.where(mid, e, torch.zeros_like(e))

    def force(self, t, d):
        f0, fd, fi = self.grids[2]
        b = torch.trunc((d - f0) * fi + 0.5).long()
        c = b.clamp(0, self.nf - 1)
        ph = (d - (f0 + c * fd)) * fi
        f = self.f[t, c + 1] * ph + self.f[t, c] * (1.0 - ph)
        return torch.where((b >= 0) & (b < self.nf), f, torch.zeros_like(f))


class _Analytic:
    """The differentiable model's functions, of theta = (sigma, eps, x0, g0, alpha) per type."""

    def __init__(self, theta, prm):
        sig, eps, self.x0, self.g0, self.al = theta.unbind(1)
        self.sts, self.ets = 0.5 * (sig + prm.sig_s), torch.sqrt(eps * prm.eps_s)
        self.rlo = torch.maximum(self.x0 - torch.sqrt(self.g0 / self.al), prm.core * self.sts)
        self.rhi = self.x0 + torch.sqrt((self.g0 - 1.0) / self.al)
        self.c, self.delta = _f64(prm.camp), prm.delta

    def _switch(self, t, d):
        z = ((d - self.rlo[t]) / self.delta + 1.0).clamp(0.0, 1.0)
        return z * z * (3.0 - 2.0 * z)

    def g_and_e(self, t, d):
        s, u = self._switch(t, d), d - self.x0[t]
        g = s * (self.g0[t] - self.al[t] * u * u).clamp(min=0.0)
        return torch.where(d < self.rhi[t], g, torch.ones_like(g)), self.c[t] * torch.exp(-0.5 * u * u) * s

    def force(self, t, d):
        r6 = (self.sts[t] / d) ** 6
        return 24.0 * self.ets[t] / d * (2.0 * r6 * r6 - r6) * self._switch(t, d)


def _isspa(x32, q, types, rmax, fns, n_mc, box, seed, step, sys_id):
    """(lj, pol, cdd) forces [n, 3] of one window."""
    k = _constants()
    n = x32.shape[0]
    t = _i64(types)
    rm32 = _f32(rmax)
    r2 = (rm32 * rm32).double()
    vt = _f64([np.float32(4.0 / 3.0 * float(np.float32(3.1415926535)) * float(r) ** 3 * 0.0074 / n_mc)
               for r in np.asarray(rmax, np.float32)])[t]
    p32, own = _points(x32, rm32[t], n_mc, seed, step, sys_id)
    piece = max(1, _PAIRS // n)
    lj, pol, cdd = (torch.zeros((n, 3), dtype=torch.float64, device=_DEV) for _ in range(3))
    for a in range(0, p32.shape[0], piece):
        p = p32[a:a + piece]
        r, d2f = _separations(p, x32, box)
        rr = r[0] * r[0] + r[1] * r[1] + r[2] * r[2]
        d = torch.sqrt(rr)
        inside = d2f <= r2[t[own[a:a + piece]]][:, None]
        # field of the atoms at the points
        s = q[None, :] / (rr * d)
        so = torch.where(inside, torch.zeros_like(s), s)
        fac, et = fns.g_and_e(t[None, :].expand_as(d)[inside], d[inside])
        ein = torch.zeros_like(s).masked_scatter(inside, et / d[inside] - k["e0"] * s[inside])
        ee0 = torch.stack([-k["e0"] * (so * c).sum(1) for c in r], 1)
        ee = ee0 + torch.stack([(ein * c).sum(1) for c in r], 1)
        ok = fac > 0.0
        lg = torch.zeros_like(s).masked_scatter(inside, torch.log(torch.where(ok, fac, torch.ones_like(fac))))
        dead = torch.zeros_like(inside).masked_scatter(inside, ~ok).any(1)
        cnt = inside.sum(1).double()
        g = torch.where(dead, torch.zeros_like(cnt), torch.exp(lg.sum(1)))
        del s, so, ein, lg
        # orientational moments of the solvent at the points
        sq = (ee * ee).sum(1)
        some = sq > 0.0  # uncharged atoms alone: no field, no direction
        mag = torch.where(some, torch.sqrt(torch.where(some, sq, torch.ones_like(sq))), torch.zeros_like(sq))
        eh = torch.where(some, 1.0 / torch.where(some, mag, torch.ones_like(sq)), torch.zeros_like(sq))[:, None] * ee
        m1, m2, m3 = _moments(mag)
        w = g / cnt
        a1, a2, a3 = k["p0"] * m1 * w, k["q0"] * m2 * w, k["o0"] * m3 * w
        ec = (k["p0"] / cnt)[:, None] * ee0
        # force of the points on the atoms
        ir = 1.0 / d
        u = (eh[:, 0:1] * r[0] + eh[:, 1:2] * r[1] + eh[:, 2:3] * r[2]) * ir
        p2 = 7.5 * u * u - 1.5
        p3 = (17.5 * u * u - 7.5) * u
        i3 = ir * ir * ir
        i4 = i3 * ir
        al = i4 * (3.0 * a1[:, None] * u + ir * (a2[:, None] * p2 + ir * a3[:, None] * p3))
        kk = i3 * a1[:, None] + i4 * (3.0 * u * a2[:, None] + ir * p2 * a3[:, None])
        del u, p2, p3
        inr = d2f <= r2[t][None, :]
        er = ec[:, 0:1] * r[0] + ec[:, 1:2] * r[1] + ec[:, 2:3] * r[2]
        zero = torch.zeros_like(i3)
        c5, c3 = torch.where(inr, zero, er * i4 * ir), torch.where(inr, zero, i3 / 3.0)
        fl = torch.zeros_like(i3).masked_scatter(
            inr, fns.force(t[None, :].expand_as(d)[inr], d[inr]) * ir[inr])
        fl = fl * w[:, None]
        qv = (-q * vt)[:, None]
        pol = pol + qv * torch.stack([(al * r[c] - kk * eh[:, c:c + 1]).sum(0) for c in range(3)], 1)
        cdd = cdd + qv * torch.stack([(c5 * r[c] - c3 * ec[:, c:c + 1]).sum(0) for c in range(3)], 1)
        lj = lj - vt[:, None] * torch.stack([(fl * r[c]).sum(0) for c in range(3)], 1)
    return lj, pol, cdd


def _excluded(prefix, lst, a0, n):
    """Excluded pairs (i, j) of atoms [a0, a0 + n), both orders, window-local."""
    out = []
    for i in range(a0, a0 + n):
        start = int(prefix[i - 1]) if i else 0
        for j in lst[start:int(prefix[i])]:
            if i < j < a0 + n:
                out += [(i - a0, int(j) - a0), (int(j) - a0, i - a0)]
    return _i64(np.array(out, np.int64).reshape(-1, 2))


def _nonbond(x32, q, ityp, pa, pb, excl, radius, box):
    """(lj, coul, pair) forces [n, 3] of one window; pa, pb [T, T]; excl pairs."""
    n = x32.shape[0]
    fep = 1.0 - 1.0 / _constants()["ep"]
    t = _i64(ityp)
    rad = _f64(radius)
    out = [torch.zeros((n, 3), dtype=torch.float64, device=_DEV) for _ in range(3)]
    piece = max(1, _PAIRS // n)
    for a in range(0, n, piece):
        i = torch.arange(a, min(n, a + piece), device=_DEV)
        r, d2f = _separations(x32[i], x32, box)
        m = len(i)
        own = i[:, None] == torch.arange(n, device=_DEV)[None, :]
        rr = torch.where(own, torch.ones_like(d2f), r[0] * r[0] + r[1] * r[1] + r[2] * r[2])
        d = torch.sqrt(rr)
        keep = torch.ones((m, n), dtype=torch.bool, device=_DEV)
        if len(excl):
            e = excl[(excl[:, 0] >= a) & (excl[:, 0] < a + m)]
            keep[e[:, 0] - a, e[:, 1]] = False
        keep &= ~own
        zero = torch.zeros_like(d)
        i6 = 1.0 / rr ** 3
        qq = q[i][:, None] * q[None, :]
        A, B = pa[t[i][:, None], t[None, :]], pb[t[i][:, None], t[None, :]]
        lj = torch.where(keep, (12.0 * A * i6 - 6.0 * B) * i6 / rr, zero)
        co = torch.where(keep, qq / (rr * d), zero)
        far = -2.0 * fep / 3.0 / (rr * d)
        near = -fep / (3.0 * rad ** 3) + fep / (8.0 * rad ** 4) * d
        pr = torch.where(own, zero, qq * torch.where(d > 2.0 * rad[None, :], far, near))
        for o, s in zip(out, (lj, co, pr)):
            o[a:a + m] = torch.stack([(s * r[c]).sum(1) for c in range(3)], 1)
    return out


def _pair_tables(s):
    T = s.n_lj_types
    p = np.asarray(s.nbparm).reshape(T, T)
    return _f64(s.lj_a[p]), _f64(s.lj_b[p])


def _mi(a, b, box):
    d = a[:, :3] - b[:, :3]
    h = float(np.float32(0.5) * np.float32(box))
    img = (d > h).double() - (d < -h).double()
    return a[:, :3].double() - b[:, :3].double() - img * float(np.float32(box))


def _dot(a, b):
    return (a * b).sum(1)


def _bonded(s, x, f):
    """Adds the bond, angle, dihedral and scaled 1-4 forces to f; five energies."""
    L = s.lbox
    e = []
    b, pr = _i64(s.bond_atoms), _f64(s.bond_params)
    pr = pr[b[:, 2]]
    r = _mi(x[b[:, 0]], x[b[:, 1]], L)
    d = torch.sqrt(_dot(r, r))
    fb = (pr[:, 0] * (pr[:, 1] / d - 1.0))[:, None] * r
    f.index_add_(0, b[:, 0], fb).index_add_(0, b[:, 1], -fb)
    e.append((0.5 * pr[:, 0] * (d - pr[:, 1]) ** 2).sum())
    a, pr = _i64(s.angle_atoms), _f64(s.angle_params)
    pr = pr[a[:, 3]]
    r1, r2 = _mi(x[a[:, 0]], x[a[:, 1]], L), _mi(x[a[:, 1]], x[a[:, 2]], L)
    c11, c22, c12 = _dot(r1, r1), _dot(r2, r2), _dot(r1, r2)
    th = torch.acos((-c12 / torch.sqrt(c11 * c22)).clamp(-1.0, 1.0)) - pr[:, 1]
    fa = (pr[:, 0] * th / torch.sqrt(c11 * c22 - c12 * c12))[:, None]
    f1 = fa * ((c12 / c11)[:, None] * r1 - r2)
    f3 = fa * (r1 - (c12 / c22)[:, None] * r2)
    f.index_add_(0, a[:, 0], f1).index_add_(0, a[:, 2], f3).index_add_(0, a[:, 1], -f1 - f3)
    e.append((0.5 * pr[:, 0] * th * th).sum())
    q4, ty = _i64(s.dih_atoms), _i64(s.dih_types)
    ty = ty.long()
    pair = (q4[:, 2] > 0) & (q4[:, 3] > 0)
    i, j, k, l = q4[:, 0], q4[:, 1], q4[:, 2].abs(), q4[:, 3].abs()
    pr, sc = _f64(s.dih_params)[ty], _f64(s.sc14)[ty]
    r12, r23, r34 = _mi(x[i], x[j], L), _mi(x[j], x[k], L), _mi(x[k], x[l], L)
    c11, c22, c33 = _dot(r12, r12), _dot(r23, r23), _dot(r34, r34)
    c12, c23, c13 = _dot(r12, r23), _dot(r23, r34), _dot(r12, r34)
    t1, t2, t3 = c13 * c22 - c12 * c23, c11 * c23 - c12 * c13, c12 * c12 - c11 * c22
    t4, t5 = c22 * c33 - c23 * c23, c13 * c23 - c12 * c33
    bb = torch.sqrt(-t3 * t4)
    phi = torch.acos((-t1 / bb).clamp(-1.0, 1.0))
    fd = pr[:, 0] * pr[:, 1] * torch.sin(pr[:, 0] * phi - pr[:, 2]) * c22 / (torch.sin(phi) * bb)
    f1 = (fd / t3)[:, None] * (t1[:, None] * r12 + t2[:, None] * r23 + t3[:, None] * r34)
    f4 = (-fd / t4)[:, None] * (t4[:, None] * r12 + t5[:, None] * r23 - t1[:, None] * r34)
    a12, a23 = (c12 / c22)[:, None], (c23 / c22)[:, None]
    f.index_add_(0, i, f1).index_add_(0, j, -(1.0 + a12) * f1 + a23 * f4)
    f.index_add_(0, k, a12 * f1 - (1.0 + a23) * f4).index_add_(0, l, f4)
    e.append((pr[:, 1] * (1.0 + torch.cos(pr[:, 0] * phi - pr[:, 2]))).sum())
    i, l, sc = i[pair], l[pair], sc[pair]
    pa, pb = _pair_tables(s)
    it = _i64(s.ityp)
    A, B = pa[it[i], it[l]], pb[it[i], it[l]]
    r = _mi(x[i], x[l], L)
    rr = _dot(r, r)
    i6 = 1.0 / rr ** 3
    qq = x[i, 3].double() * x[l, 3].double()
    ft = qq / (rr * torch.sqrt(rr) * sc[:, 0]) + i6 * (12.0 * A * i6 - 6.0 * B) / (sc[:, 1] * rr)
    f.index_add_(0, i, ft[:, None] * r).index_add_(0, l, -ft[:, None] * r)
    e.append((qq / (torch.sqrt(rr) * sc[:, 0])).sum())
    e.append(((A * i6 * i6 - B * i6) / sc[:, 1]).sum())
    return torch.stack(e)


def _restraint(us, box, x, f):
    at = _i64(us.atom_list)
    m = _f64(us.mass)[:, None]
    g1 = at[:, 1] == 1
    pos = x[at[:, 0], :3].double() * m
    dv = pos[~g1].sum(0) - pos[g1].sum(0)
    dv = dv - box * ((dv > 0.5 * box).double() - (dv < -0.5 * box).double())
    d = torch.sqrt((dv * dv).sum())
    pre = torch.where(g1, us.k, -us.k).double()[:, None] * (d - us.x0) * m / d
    f.index_add_(0, at[:, 0], pre * dv[None, :])


def _parts(s):
    """(first atom, atoms, system id, box, restraint) of every window."""
    if getattr(s, "windows", None) is None:
        return [(0, s.n_atoms, 0, s.lbox, s.us)]
    a0 = np.concatenate([[0], np.cumsum(s.windows)[:-1]])
    return [(int(a), int(n), int(i), float(L), u) for a, n, i, L, u in
            zip(a0, s.windows, s.window_sys, s.window_lbox, s.restraints)]


class _Exact:
    """Forces and steps of one system in 64 bits, its state rounded to FP32 after each step."""

    def __init__(self, s):
        self.s, self.fns = s, _Tables(s.isspa)
        self.x, self.v = _f32(s.xyzq), _f32(s.vel)
        self.pa, self.pb = _pair_tables(s)
        self.parts = _parts(s)
        self.excl = [_excluded(s.nexcl_prefix, s.excl_list, a, n) for a, n, _, _, _ in self.parts]

    def isspa(self, step):
        s, it = self.s, self.s.isspa
        out = [_isspa(self.x[a:a + n, :3], self.x[a:a + n, 3].double(), it.isspa_type[a:a + n],
                      it.rmax, self.fns, s.n_mc, L, int(s.seed), step, w)
               for a, n, w, L, _ in self.parts]
        return [torch.cat(c) for c in zip(*out)]

    def nonbond(self):
        s, it = self.s, self.s.isspa
        out = [_nonbond(self.x[a:a + n, :3], self.x[a:a + n, 3].double(), s.ityp[a:a + n], self.pa,
                        self.pb, ex, it.rmax[it.isspa_type[a:a + n]], L)
               for (a, n, _, L, _), ex in zip(self.parts, self.excl)]
        return [torch.cat(c) for c in zip(*out)]

    def total(self, step):
        f = sum(self.isspa(step)) + sum(self.nonbond())
        e = _bonded(self.s, self.x, f) if len(self.s.bond_atoms) else None
        for _, _, _, L, us in self.parts:
            if us is not None:
                _restraint(us, L, self.x, f)
        return f, e

    def integrate(self, f, step):
        s = self.s
        m = self.v[:, 3:4].double()
        thr = int(float(np.float32(s.pnu)) * 4294967296.0)
        v, dt = self.v[:, :3].double(), s.dt
        il = torch.cat([torch.arange(n, device=_DEV) for _, n, _, _, _ in self.parts])
        kick = v + f * dt / m
        hit, new = [], []
        for a, n, w, _, _ in self.parts:
            o = _philox(il[a:a + n], 1, 0, step, w, int(s.seed))
            z = _philox(il[a:a + n], 1, 1, step, w, int(s.seed))
            u = [(((k >> 8) + 1 - c).double()) * 2.0 ** -24 for k, c in zip(z, (0, 1, 0, 1))]
            ra, rb = torch.sqrt(-2.0 * torch.log(u[0])), torch.sqrt(-2.0 * torch.log(u[2]))
            p1, p2 = 2.0 * math.pi * u[1], 2.0 * math.pi * u[3]
            hit.append(o[0] < thr)
            new.append(torch.stack([ra * torch.cos(p1), ra * torch.sin(p1), rb * torch.cos(p2)], 1))
        drawn = torch.cat(new) * torch.sqrt(s.kT / m) + f * dt / (2.0 * m)
        v = torch.where(torch.cat(hit)[:, None], drawn, kick)
        x = self.x[:, :3].double() + v * dt
        box = torch.cat([torch.full((n, 1), float(L), device=_DEV, dtype=torch.float64)
                         for _, n, _, L, _ in self.parts])
        x = torch.where(x > box, x - box, torch.where(x < 0.0, x + box, x))
        self.v = torch.cat([v.float(), self.v[:, 3:4]], 1)
        self.x = torch.cat([x.float(), self.x[:, 3:4]], 1)
        return torch.cat([x, self.x[:, 3:4].double()], 1), torch.cat([v, m], 1)


def _four(f):
    return torch.cat([f, torch.zeros_like(f[:, :1])], 1)


def _match_exact(case, seed):
    s, prm, theta, q, target = _match_inputs(case, seed)
    theta, q = _f64(theta).requires_grad_(), _f64(q).requires_grad_()
    target = _f64(target)
    norm = float((target ** 2).mean())
    it, x = s.isspa, _f32(s.xyzq)
    gt, gq = torch.zeros_like(theta), torch.zeros_like(q)
    forces, loss = [], 0.0
    for a, n, w, L, _ in _parts(s):
        fns = _Analytic(theta, prm)
        sig, eps = theta[:, 0], theta[:, 1]
        s6 = (0.5 * (sig[:, None] + sig[None, :])) ** 6
        e4 = 4.0 * torch.sqrt(eps[:, None] * eps[None, :])
        qw, ty = q[a:a + n], it.isspa_type[a:a + n]
        ex = _excluded(s.nexcl_prefix, s.excl_list, a, n)
        f = sum(_isspa(x[a:a + n, :3], qw, ty, it.rmax, fns, s.n_mc, L, int(s.seed), 0, w))
        f = f + sum(_nonbond(x[a:a + n, :3], qw, ty, e4 * s6 * s6, e4 * s6, ex, it.rmax[ty], L))
        part = ((f - target[a:a + n]) ** 2).sum() / target.numel() / norm
        dt, dq = torch.autograd.grad(part, [theta, q])
        gt, gq, loss = gt + dt, gq + dq, loss + part.detach()
        forces.append(f.detach())
    return {"forces": torch.cat(forces), "loss": loss, "grad_theta": gt, "grad_q": gq}


def exact(case, seed):
    kind = case["kind"]
    if kind == "match":
        return _match_exact(case, seed)
    with torch.no_grad():
        s = _windows(case, seed) if kind == "batch" else _system(case, seed)
        m = _Exact(s)
        if kind == "isspa":
            return {"f": _four(sum(m.isspa(0)))}
        if kind == "nonbond":
            return {"f": _four(sum(m.nonbond()))}
        if kind == "components":
            return {**dict(zip(("isspa_lj", "isspa_pol", "isspa_cdd"), m.isspa(0))),
                    **dict(zip(("nonbond_lj", "nonbond_coul", "nonbond_pair"), m.nonbond()))}
        for step in range(case.get("steps", 1)):
            f, e = m.total(step)
            x, v = m.integrate(f, step)
        out = {"x": x, "v": v, "f": _four(f)}
        if kind == "loop":
            out["energies"] = e
        return out
