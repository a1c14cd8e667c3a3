"""The measured workloads of the ring-polymer engine, through its Python entry points.

Three groups, as the two drivers use the package:

* ``batch``  PIMD thermodynamic integration: a ``Batch`` of trajectories (lambda nodes x
  replicas x bead counts) after ``set_path`` / ``init_path``; a pass is one ``run`` of
  ``steps`` steps with its TI readout (and, for a small job, every trajectory's x and p, as
  a run writes its restart files).
* ``chain``  one trajectory at a time, as a caller of the reference's ``verletint`` steps it:
  state in, ``propagate_pimd_pile``, state out.
* ``action`` / ``hvp`` / ``search`` / ``logdet``  the ring-polymer instanton: the action and
  its gradient through ``ring_action`` under torch.autograd, its Hessian-vector product, the
  L-BFGS search and the fluctuation determinant, for many chains of uneven length at once.

``exact`` repeats each pass in plain float64 torch from the defining formulas: the
reference's dense normal-mode transform (with its truncated literal of pi), the A-O-A step,
its Philox draws, and block factorisations for the determinant.
"""
import math
import os
import sys

import numpy as np
import torch

_PY = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                   "pimd-tunneling_amd", "python")
if _PY not in sys.path:
    sys.path.insert(0, _PY)

from rptunnel import Batch, Chain, Pes, Ring, specs, ti  # noqa: E402
from rptunnel.autograd import ring_action  # noqa: E402

PI_REF = 3.14159265358979
TAU, DT, GAMMA, BETA = 20.0, 1.0, 1.0e-3, 2000.0
LANGEVIN, ANDERSEN = 2, 1
DEV = "cuda"


# --------------------------------------------------------------------------- the cases
def _batch(name, pes, ns, nodes, reps, steps, thermostat=LANGEVIN, noutput=1, cayley=False,
           states=False):
    return dict(name=name, path="batch", pes=pes, ns=",".join(str(n) for n in ns), nodes=nodes,
                reps=reps, steps=steps, thermostat=thermostat, noutput=noutput, cayley=cayley,
                states=states)


def _rings(name, path, pes, chains, nlo, nhi, **more):
    return dict(name=name, path=path, pes=pes, chains=chains, nlo=nlo, nhi=nhi, **more)


def listed():
    return [
        # the smallest call: one short trajectory of one chain, state in and out, as the
        # drop-in for the reference's per-trajectory integrator is called
        dict(name="chain_evb27_n32", path="chain", pes="evb", n=32, steps=8, cayley=False),
        # a small TI job of the 1D quartic double well, 11 nodes x 8 replicas: fewer
        # trajectories than the GPU has compute units
        _batch("ti_quartic_n64", "quartic", [64], 11, 8, 64),
        # a small TI job of the 27-dof EVB double well at N = 32
        _batch("ti_evb27_n32", "evb", [32], 11, 4, 64),
        # a convergence study in the bead count with odd and ragged N and the Cayley step,
        # one replica; x and p of every trajectory come back, as for its restart files
        _batch("ti_evb27_ragged", "evb", [17, 45, 99, 150, 251], 11, 1, 24, cayley=True,
               states=True),
        # the 2D coupled double well in bulk: 65,536 trajectories of 128 beads
        _batch("ti_coupled2d_n128", "coupled2d", [128], 16, 4096, 8),
        # the production TI of the EVB double well: six bead counts, 33,792 trajectories
        _batch("ti_evb27_mix", "evb", [32, 64, 96, 128, 192, 256], 11, 512, 8),
        # the same surface under the Andersen thermostat
        _batch("ti_evb27_andersen", "evb", [64, 256], 11, 512, 8, thermostat=ANDERSEN, noutput=5),
        # the water hexamer (54 dof), its path the rotation that exchanges two hydrogens
        _batch("ti_water6_n128", "water6", [128], 11, 1024, 8),
        # instantons: 256 chains of 64 to 1024 beads; action and gradient, and the
        # Hessian-vector product of a second-order method on fewer, shorter chains
        _rings("action_evb27", "action", "evb", 256, 64, 1024),
        _rings("hvp_evb27", "hvp", "evb", 64, 64, 256),
        # the first iterations of the spring-preconditioned instanton search
        _rings("search_evb27", "search", "evb", 128, 64, 512, iters=10),
        # lndetJ at kinked chains: log-determinant without the lowest eigenvalue
        _rings("logdet_evb27", "logdet", "evb", 256, 64, 1024),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["batch", "batch", "batch", "batch", "chain", "action", "hvp", "search", "logdet"])
    if kind == "batch":
        pes = rng.choice(["evb", "evb", "quartic", "coupled2d", "water6"])
        ns = [_log(rng, 12, 128 if pes == "water6" else 256) for _ in range(rng.choice([1, 1, 2, 3]))]
        steps = rng.choice([8, 16, 24])
        # bead-steps x dof of the listed bulk cases at most
        most = 1.2e9 / (steps * sum(ns) * {"quartic": 6, "coupled2d": 8, "evb": 27, "water6": 100}[pes])
        nodes = rng.choice([5, 8, 11, 16])
        reps = _log(rng, 1, max(1, min(2048, most / nodes)))
        andersen = rng.random() < 0.25
        c = _batch("", pes, sorted(set(ns)), nodes, reps, steps,
                   thermostat=ANDERSEN if andersen else LANGEVIN,
                   noutput=rng.choice([3, 5, 20]) if andersen else 1, cayley=rng.random() < 0.25,
                   states=nodes * reps <= 16)
    elif kind == "chain":
        c = dict(path="chain", pes=rng.choice(["evb", "coupled2d", "quartic", "water6"]),
                 n=_log(rng, 12, 128), steps=_log(rng, 4, 24), cayley=rng.random() < 0.25)
    else:
        nhi = _log(rng, 80, {"action": 1024, "hvp": 512, "search": 512, "logdet": 768}[kind])
        c = _rings("", kind, "evb", _log(rng, 4, {"action": 256, "hvp": 128, "search": 128,
                                                   "logdet": 192}[kind]), max(16, nhi // 8), nhi)
        if kind == "search":
            c["iters"] = rng.randint(6, 12)
    c.pop("name", None)
    return c


# --------------------------------------------------------------------------- inputs
def _spec(name):
    return {"quartic": specs.quartic, "coupled2d": specs.coupled2d, "evb": specs.evb,
            "water6": lambda: specs.water_cluster(nmol=6)}[name]()


def _ns(case):
    return [int(v) for v in str(case["ns"]).split(",")]


def _path(case, sp):
    """(lampath, path (ndof, npath)): the straight line, or the water hexamer's rotation."""
    if case["pes"] == "water6":
        path = np.ascontiguousarray(sp.extra["path"].T)
        return specs.arc_lampath(path), path
    return specs.linear_path(sp.well1, sp.well2, npath=2)


def _spline(x, path):
    """Natural cubic spline of every row of path: second derivatives (ndof, npath)."""
    n = len(x)
    A, r, h = np.eye(n), np.zeros((n, path.shape[0])), np.diff(x)
    for i in range(1, n - 1):
        A[i, i - 1:i + 2] = h[i - 1], 2.0 * (h[i - 1] + h[i]), h[i]
        r[i] = 6.0 * ((path[:, i + 1] - path[:, i]) / h[i] - (path[:, i] - path[:, i - 1]) / h[i - 1])
    return np.linalg.solve(A, r).T


def _splint(x, path, y2, at, slope=False):
    """The spline (or its derivative) of every row at the points `at`: (len(at), ndof)."""
    at = np.asarray(at, float)
    k = np.clip(np.searchsorted(x, at, side="right") - 1, 0, len(x) - 2)
    h = x[k + 1] - x[k]
    a, b = (x[k + 1] - at) / h, (at - x[k]) / h
    p0, p1, s0, s1 = path[:, k], path[:, k + 1], y2[:, k], y2[:, k + 1]
    if slope:
        return ((p1 - p0) / h - (3 * a * a - 1) / 6 * h * s0 + (3 * b * b - 1) / 6 * h * s1).T
    return (a * p0 + b * p1 + ((a ** 3 - a) * s0 + (b ** 3 - b) * s1) * h * h / 6).T


def _polymers(case, sp):
    lampath, path = _path(case, sp)
    y2 = _spline(lampath, path)
    xi, _ = ti.gauleg(0.0, 1.0, case["nodes"])
    ends, grads = _splint(lampath, path, y2, xi), _splint(lampath, path, y2, xi, slope=True)
    start = np.ascontiguousarray(path[:, 0])
    pols, stream = [], 0
    for n in _ns(case):
        for i, x in enumerate(xi):
            b, d = np.ascontiguousarray(ends[i]), np.ascontiguousarray(grads[i])
            for _ in range(case["reps"]):
                pols.append(dict(n=n, betan=BETA / (n + 1), xi=float(x), a=start, b=b, dbdl=d,
                                 stream=stream))
                stream += 1
    return pols, lampath, path, y2


def _chain_inputs(case, seed):
    """One chain's x and p, its ends and db/dlambda: the path up to lambda = 1/2 with the
    spread of a thermal chain."""
    sp = _spec(case["pes"])
    n = case["n"]
    rng = np.random.default_rng(seed)
    lampath, path = _path(case, sp)
    y2 = _spline(lampath, path)
    x = _splint(lampath, path, y2, 0.5 * np.arange(n) / (n - 1)).T
    x = x + 0.01 * rng.standard_normal(x.shape)
    m = np.repeat(sp.mass, sp.ndim)[:, None]
    i = np.arange(1, n + 1)
    bn = BETA / (n + 1)
    lam = 2.0 * np.sin(i * np.pi / (2 * n + 2)) / bn
    T = np.sin(np.outer(i, i) * np.pi / (n + 1)) * np.sqrt(2.0 / (n + 1))
    p = (np.sqrt(m / bn) * lam * TAU * rng.standard_normal(x.shape)) @ T
    a, b = path[:, 0].copy(), _splint(lampath, path, y2, [0.5])[0]
    return sp, x, p, a, b, _splint(lampath, path, y2, [0.5], slope=True)[0]


def _ring_inputs(case, seed):
    """Chain lengths (a case's own), betan = beta / N with beta in [1000, 8000], and the chains:
    kinks that leave the two wells with exponential tails, as instantons do, and a little noise.  No bead
    sits on the barrier's top, so every chain's Hessian is positive definite, with the paired
    low eigenvalues of its two halves."""
    sp = _spec(case["pes"])
    lengths = np.random.default_rng([case["chains"], case["nlo"], case["nhi"]])
    ns = [int(v) for v in lengths.integers(case["nlo"], case["nhi"] + 1, case["chains"])]
    rng = np.random.default_rng(seed)
    betan = [float(b) / n for b, n in zip(rng.uniform(1000.0, 8000.0, len(ns)), ns)]
    chains = []
    for n, bn in zip(ns, betan):
        mid = 0.5 * (n - 1) + rng.uniform(-0.4, 0.4) * (n > 32)
        t = (np.arange(n) - mid) * bn
        f = 0.15 * np.exp(-np.abs(t) / 60.0)
        f = np.where(t < 0, f, 1.0 - f)
        x = np.outer(sp.well1, 1.0 - f) + np.outer(sp.well2, f)
        chains.append(x + 0.004 * rng.standard_normal(x.shape))
    return sp, ns, betan, chains


def _flat(chains):
    return torch.from_numpy(np.concatenate([c.reshape(-1) for c in chains])).to(DEV)


def prepare(case, seed):
    if case["path"] == "batch":
        sp = _spec(case["pes"])
        pes = Pes(sp)
        pols, lampath, path, _ = _polymers(case, sp)
        b = Batch(pes, sp.mass, pols, TAU, DT, GAMMA, thermostat=case["thermostat"],
                  noutput=case["noutput"], cayley=case["cayley"], seed=seed)
        b.set_path(lampath, path)
        b.init_path()
        return dict(case=case, pes=pes, batch=b)
    if case["path"] == "chain":
        sp, x, p, a, b, dbdl = _chain_inputs(case, seed)
        pes = Pes(sp)
        ch = Chain(pes, case["n"], sp.mass, BETA / (case["n"] + 1), TAU, DT, GAMMA, a, b,
                   cayley=case["cayley"])
        ch.set_rng(seed, 3)
        return dict(case=case, pes=pes, chain=ch, x=x, p=p, dbdl=dbdl)
    sp, ns, betan, chains = _ring_inputs(case, seed)
    pes = Pes(sp)
    ring = Ring(pes, sp.mass, ns, betan, sp.well1, sp.well2)
    st = dict(case=case, pes=pes, ring=ring, chains=chains)
    if case["path"] in ("action", "hvp"):
        st["x"] = _flat(chains).requires_grad_(True)
        st["v"] = torch.randn(st["x"].numel(), dtype=torch.float64, device=DEV,
                              generator=torch.Generator(DEV).manual_seed(seed))
    if case["path"] == "search":
        ring.set_preconditioner(0.05)
    if case["path"] == "logdet":
        ring.set_x(chains)
    return st


# --------------------------------------------------------------------------- one pass
def run(state):
    case = state["case"]
    if case["path"] == "batch":
        b = state["batch"]
        b.run(case["steps"])
        sums, count, nreinit = b.ti_readout()
        out = dict(sums=sums, count=count, nreinit=nreinit, cursor=b.cursors())
        if case["states"]:
            xp = [b.get_state(k) for k in range(b.npoly)]
            out["x"] = np.concatenate([x.reshape(-1) for x, _ in xp])
            out["p"] = np.concatenate([p.reshape(-1) for _, p in xp])
        return out
    if case["path"] == "chain":
        ch = state["chain"]
        ch.set_state(state["x"], state["p"])
        dhdr, _ = ch.propagate_pimd_pile(case["steps"], state["dbdl"])
        x, p = ch.get_state()
        return dict(dhdr=dhdr, x=x, p=p)
    ring = state["ring"]
    if case["path"] == "action":
        u = ring_action(state["x"], ring)
        (g,) = torch.autograd.grad(u.sum(), state["x"])
        return dict(u=u.detach(), g=g)
    if case["path"] == "hvp":
        u = ring_action(state["x"], ring)
        (g,) = torch.autograd.grad(u.sum(), state["x"], create_graph=True)
        (hv,) = torch.autograd.grad(g, state["x"], state["v"])
        return dict(u=u.detach(), g=g.detach(), hv=hv)
    if case["path"] == "search":
        x, act, it, st = ring.instanton(state["chains"], pgtol=1e-5, factr=1e6, m=8,
                                        maxiter=case["iters"])
        return dict(x=np.concatenate([c.reshape(-1) for c in x]), action=act, iters=it, status=st)
    ld, nneg, eta = ring.logdet(singlewell=False, skip_lowest=True)
    return dict(logdet=ld, nneg=nneg, eta=eta)


# --------------------------------------------------------------------------- algorithmic work
def _pes_flops(name, d):
    """Of one bead's gradient."""
    return {"quartic": 8.0 * d, "coupled2d": 20.0, "evb": 8.0 * d * d + 26.0 * d,
            "water6": 6 * 120.0 + 135 * 35.0}[name]


def work(case):
    d = {"quartic": 1, "coupled2d": 2, "evb": 27, "water6": 54}[case["pes"]]
    wp = _pes_flops(case["pes"], d)
    if case["path"] in ("batch", "chain"):
        ns = _ns(case) if case["path"] == "batch" else [case["n"]]
        pols = case["nodes"] * case["reps"] if case["path"] == "batch" else 1
        beads = float(sum(ns)) * pols * case["steps"]
        # per bead-step: the force, the A-O-A step (its normals and its recurrences along
        # the chain), and for Langevin one folded transform of the noise
        sq = float(sum(n * n for n in ns)) * pols * case["steps"]
        langevin = case.get("thermostat", LANGEVIN) == LANGEVIN
        flops = beads * (wp + 60.0 * d) + (d * sq if langevin else 0.0)
        return dict(bytes=32.0 * d * sum(ns) * pols, flops=flops)
    beads = float(case["chains"]) * 0.5 * (case["nlo"] + case["nhi"])
    if case["path"] == "action":
        return dict(bytes=16.0 * d * beads, flops=beads * (wp + 10.0 * d))
    if case["path"] == "hvp":
        return dict(bytes=32.0 * d * beads, flops=beads * (3.0 * wp + 20.0 * d))
    if case["path"] == "search":
        return dict(bytes=16.0 * d * beads * (1.0 + case["iters"]),
                    flops=beads * (1.0 + case["iters"]) * (wp + 80.0 * d))
    # the Hessian blocks, one symmetric elimination of each, and a few block solves
    return dict(bytes=8.0 * d * beads, flops=beads * (2.0 * d * wp + 2.0 * d ** 3 + 40.0 * d * d))


# --------------------------------------------------------------------------- float64 references
_M32 = 0xFFFFFFFF


def _philox(block, stream, seed):
    """Philox4x32-10: counter (block, stream), key seed -> the two 53-bit uniforms of a block."""
    c = [block & _M32, (block >> 32) & _M32, stream & _M32, (stream >> 32) & _M32]
    k0, k1 = seed & _M32, (seed >> 32) & _M32
    for r in range(10):
        if r:
            k0, k1 = (k0 + 0x9E3779B9) & _M32, (k1 + 0xBB67AE85) & _M32
        p0, p1 = c[0] * 0xD2511F53, c[2] * 0xCD9E8D57
        c = [((p1 >> 32) & _M32) ^ c[1] ^ k0, p1 & _M32, ((p0 >> 32) & _M32) ^ c[3] ^ k1, p0 & _M32]
    u = [((c[2 * j + 1] << 21) | (c[2 * j] >> 11)).to(torch.float64) for j in (0, 1)]
    return [(v + 0.5) * 2.0 ** -53 for v in u]


def _normals(seed, stream, index):
    """Draw `index` of each stream (Box-Muller on the block index // 2)."""
    u0, u1 = _philox(index >> 1, stream, seed)
    r, a = torch.sqrt(-2.0 * torch.log(u0)), 2.0 * math.pi * u1
    return torch.where((index & 1) == 0, r * torch.cos(a), r * torch.sin(a))


def _poisson(seed, stream, index, mean):
    """Poisson interval `index` of each stream: inversion below mean 16, else rounded normal."""
    high = torch.tensor(-2 ** 63, dtype=torch.int64, device=stream.device)
    u0, u1 = _philox(index, stream ^ high, seed)
    if mean >= 16.0:
        z = torch.sqrt(-2.0 * torch.log(u0)) * torch.cos(6.283185307179586 * u1)
        return torch.clamp(torch.floor(mean + math.sqrt(mean) * z + 0.5), min=0.0).to(torch.int64)
    k = torch.zeros_like(index)
    pk = cdf = math.exp(-mean)
    for j in range(1, 200):
        k = torch.where(u0 > cdf, torch.full_like(k, j), k)
        pk *= mean / j
        cdf += pk
    return k


def _energy(sp, x):
    """V of every bead; x (..., ndof, n) -> (..., n)."""
    dp = sp.dp
    if sp.name == "quartic":
        return (dp[0] * ((x / dp[1]) ** 2 - 1.0) ** 2).sum(-2)
    if sp.name == "coupled2d":
        v0, a, m, w, c = dp
        return v0 * ((x[..., 0, :] / a) ** 2 - 1.0) ** 2 \
            + 0.5 * m * w * w * (x[..., 1, :] + c * x[..., 0, :] ** 2) ** 2
    if sp.name == "evb":
        col = [torch.as_tensor(v, device=x.device)[:, None] for v in
               (sp.extra["lam"], sp.extra["cub"], sp.well1)]
        qt = torch.as_tensor(np.ascontiguousarray(sp.extra["Q"].T), device=x.device)
        atoms = np.concatenate([3 * int(p) + np.arange(3) for p in sp.extra["perm"]])

        def well(z):
            y = torch.matmul(qt, z - col[2])
            return (0.5 * col[0] * y * y + col[1] * y ** 3).sum(-2)

        va, vb = well(x), well(x[..., torch.as_tensor(atoms, device=x.device), :])
        return 0.5 * (va + vb) - torch.sqrt(0.25 * (va - vb) ** 2 + float(dp[0]) ** 2)
    de, al, re, kb, th0, eps, sig, qh = (float(v) for v in dp)
    na = sp.natom
    r3 = x.reshape(*x.shape[:-2], na, 3, x.shape[-1])
    e = 0.0
    for o in range(0, na, 3):
        u, v = r3[..., o + 1, :, :] - r3[..., o, :, :], r3[..., o + 2, :, :] - r3[..., o, :, :]
        ru, rv = u.norm(dim=-2), v.norm(dim=-2)
        e = e + de * (1 - torch.exp(-al * (ru - re))) ** 2 + de * (1 - torch.exp(-al * (rv - re))) ** 2
        e = e + 0.5 * kb * (torch.acos((u * v).sum(-2) / (ru * rv)) - th0) ** 2
        for i in range(o, o + 3):
            for j in range(o + 3, na):
                r = (r3[..., i, :, :] - r3[..., j, :, :]).norm(dim=-2)
                e = e + qh * qh * (-2.0 if i == o else 1.0) * (-2.0 if j % 3 == 0 else 1.0) / r
                if i == o and j % 3 == 0:
                    s6 = (sig / r) ** 6
                    e = e + 4.0 * eps * (s6 * s6 - s6)
    return e


def _gradient(sp, x, chunk=512):
    out = torch.empty_like(x)
    for k in range(0, x.shape[0], chunk):
        z = x[k:k + chunk].detach().requires_grad_(True)
        (out[k:k + chunk],) = torch.autograd.grad(_energy(sp, z).sum(), z)
    return out


class _Sim:
    """The reference's step on (npoly, ndof, n) arrays: dense transforms, rotation A(dt/2) of
    every normal mode at frequency 1/tau, and the Langevin O step."""

    def __init__(self, sp, n, a, b, cayley):
        i = torch.arange(1, n + 1, dtype=torch.float64, device=DEV)
        bn = BETA / (n + 1)
        self.sp, self.n, self.bn = sp, n, bn
        self.m = torch.as_tensor(np.repeat(sp.mass, sp.ndim), device=DEV)[:, None]
        self.T = torch.sin(torch.outer(i, i) * PI_REF / (n + 1)) * math.sqrt(2.0 / (n + 1))
        self.lam = 2.0 * torch.sin(i * PI_REF / (2 * n + 2)) / bn
        s = math.sqrt(2.0 / (n + 1)) / (self.lam * bn) ** 2
        self.bv = a[..., None] * (torch.sin(i * PI_REF / (n + 1)) * s) \
            + b[..., None] * (torch.sin(n * i * PI_REF / (n + 1)) * s)
        h = 0.5 * DT
        if cayley:
            w2 = h * h / (TAU * TAU)
            self.rot = (4.0 - w2) / (4.0 + w2), 4.0 * h / (TAU * TAU * (4.0 + w2)), 4.0 * h / (4.0 + w2)
        else:
            self.rot = math.cos(h / TAU), math.sin(h / TAU) / TAU, TAU * math.sin(h / TAU)
        c1 = math.exp(-GAMMA * DT / TAU)
        self.c1sq = c1 * c1
        self.kap = TAU * math.sqrt(1.0 - c1 * c1) * math.sqrt((1.0 + c1 * c1) / bn)

    def rotate(self, q, p):
        c, sq, sp = self.rot
        w = self.m * self.lam ** 2
        return c * q + (sq / w) * p, -(sp * w) * q + c * p

    def kick(self, x, p):
        return p - DT * _gradient(self.sp, x)

    def langevin(self, x, p, z):
        p = self.kick(x, p)
        q, p = self.rotate(x @ self.T - self.bv, p @ self.T)
        p = self.c1sq * p + torch.sqrt(self.m) * self.lam * self.kap * z
        q, p = self.rotate(q, p)
        return (q + self.bv) @ self.T, p @ self.T

    def half(self, x, p):
        q, p = self.rotate(x @ self.T - self.bv, p @ self.T)
        return (q + self.bv) @ self.T, p @ self.T

    def momenta(self, z):
        return (math.sqrt(1.0 / self.bn) * torch.sqrt(self.m) * self.lam * TAU * z) @ self.T

    def draws(self, seed, stream, cursor, resample):
        """n*ndof normals of each polymer from its cursor; resamples run dim-outer."""
        d = torch.arange(self.sp.ndof, device=DEV)
        if resample:
            d = (d % self.sp.ndim) * self.sp.natom + d // self.sp.ndim
        k = d[:, None] * self.n + torch.arange(self.n, device=DEV)
        return _normals(seed, stream[:, None, None], cursor[:, None, None] + k)


def _exact_batch(case, seed):
    sp = _spec(case["pes"])
    pols, lampath, path, y2 = _polymers(case, sp)
    res = dict(sums=[], count=[], nreinit=[], cursor=[], x=[], p=[])
    for n in _ns(case):
        mine = [q for q in pols if q["n"] == n]
        ab = [torch.as_tensor(np.stack([q[k] for q in mine]), device=DEV) for k in ("a", "b", "dbdl")]
        stream = torch.tensor([q["stream"] for q in mine], dtype=torch.int64, device=DEV)
        sim = _Sim(sp, n, ab[0], ab[1], case["cayley"])
        x0 = {xi: _splint(lampath, path, y2, np.arange(n) * xi / (n - 1)).T for xi in {q["xi"] for q in mine}}
        x = torch.as_tensor(np.stack([x0[q["xi"]] for q in mine]), device=DEV)
        cursor = torch.zeros_like(stream)
        need = n * sp.ndof
        p = sim.momenta(sim.draws(seed, stream, cursor, True))
        cursor += need
        sums = torch.zeros(len(mine), dtype=torch.float64, device=DEV)
        kcur = torch.zeros_like(stream)
        acount = torch.zeros_like(stream)
        if case["thermostat"] == ANDERSEN:
            kick = _poisson(seed, stream, kcur, float(case["noutput"]))
            kcur += 1
        for _ in range(case["steps"]):
            if case["thermostat"] == LANGEVIN:
                x, p = sim.langevin(x, p, sim.draws(seed, stream, cursor, False))
                cursor += need
            else:
                acount += 1
                hit = acount >= kick
                fresh = sim.momenta(sim.draws(seed, stream, cursor, True))
                p = torch.where(hit[:, None, None], fresh, p)
                cursor += need * hit
                x, p = sim.half(x, p)
                x, p = sim.half(x, sim.kick(x, p))
                kick = torch.where(hit, _poisson(seed, stream, kcur, float(case["noutput"])), kick)
                kcur += hit
                acount *= ~hit
            sums += (sim.m[:, 0] * -x[:, :, -1] * ab[2]).sum(1)
        res["sums"].append(sums)
        res["count"].append(torch.full_like(stream, case["steps"]))
        res["nreinit"].append(torch.zeros_like(stream))
        res["cursor"].append(cursor)
        res["x"].append(x.reshape(-1))
        res["p"].append(p.reshape(-1))
    keys = list(res) if case["states"] else ["sums", "count", "nreinit", "cursor"]
    return {k: torch.cat(res[k]) for k in keys}


def _exact_chain(case, seed):
    sp, x, p, a, b, dbdl = _chain_inputs(case, seed)
    t = [torch.as_tensor(v, device=DEV)[None] for v in (x, p, a, b, dbdl)]
    sim = _Sim(sp, case["n"], t[2], t[3], case["cayley"])
    x, p = t[0], t[1]
    stream = torch.tensor([3], dtype=torch.int64, device=DEV)
    cursor, total = torch.zeros_like(stream), 0.0
    for _ in range(case["steps"]):
        x, p = sim.langevin(x, p, sim.draws(seed, stream, cursor, False))
        cursor += case["n"] * sp.ndof
        total += float((sim.m[:, 0] * -x[0, :, -1] * t[4][0]).sum())
    return dict(dhdr=total / case["steps"], x=x[0], p=p[0])


def _action(sp, x, bn, a, b):
    m = torch.as_tensor(np.repeat(sp.mass, sp.ndim), device=x.device)[:, None]
    full = torch.cat([a[:, None], x, b[:, None]], dim=1)
    return _energy(sp, x).sum() + (0.5 / bn ** 2 * m * (full[:, 1:] - full[:, :-1]) ** 2).sum()


def _exact_action(case, seed):
    sp, ns, betan, chains = _ring_inputs(case, seed)
    a, b = torch.as_tensor(sp.well1, device=DEV), torch.as_tensor(sp.well2, device=DEV)
    v = torch.randn(sum(c.size for c in chains), dtype=torch.float64, device=DEV,
                    generator=torch.Generator(DEV).manual_seed(seed))
    us, gs, hs, at = [], [], [], 0
    for bn, c in zip(betan, chains):
        x = torch.as_tensor(c, device=DEV).requires_grad_(True)
        u = _action(sp, x, bn, a, b)
        (g,) = torch.autograd.grad(u, x, create_graph=case["path"] == "hvp")
        if case["path"] == "hvp":
            (h,) = torch.autograd.grad(g, x, v[at:at + c.size].reshape(x.shape))
            hs.append(h.reshape(-1))
        at += c.size
        us.append(u.detach())
        gs.append(g.detach().reshape(-1))
    out = dict(u=torch.stack(us), g=torch.cat(gs))
    if hs:
        out["hv"] = torch.cat(hs)
    return out


def _evb_hessian(sp, x):
    """Mass-weighted potential Hessians of beads x (ndof, n): (n, ndof, ndof)."""
    q, lam, cub = (torch.as_tensor(np.ascontiguousarray(sp.extra[k]), device=x.device) for k in ("Q", "lam", "cub"))
    atoms = np.concatenate([3 * int(p) + np.arange(3) for p in sp.extra["perm"]])
    qb = torch.empty_like(q)
    qb[torch.as_tensor(atoms, device=x.device)] = q  # VB(x) = VA(Pi x): y = Q^T (Pi x - xa)
    xa = torch.as_tensor(sp.well1, device=x.device)
    v, g, h = [], [], []
    for w in (q, qb):
        y = x.T @ w - xa @ q
        v.append((0.5 * lam * y * y + cub * y ** 3).sum(1))
        g.append((lam * y + 3.0 * cub * y * y) @ w.T)
        h.append((w * (lam + 6.0 * cub * y)[:, None, :]) @ w.T)
    dl, dg = v[0] - v[1], g[0] - g[1]
    r = torch.sqrt(0.25 * dl * dl + float(sp.dp[0]) ** 2)
    f = (dl / (4.0 * r))[:, None, None]
    rr = (0.25 / r - dl * dl / (16.0 * r ** 3))[:, None, None]
    hess = (0.5 - f) * h[0] + (0.5 + f) * h[1] - rr * dg[:, :, None] * dg[:, None, :]
    im = torch.as_tensor(1.0 / np.sqrt(np.repeat(sp.mass, sp.ndim)), device=x.device)
    return hess * im[:, None] * im


def _exact_logdet(case, seed):
    """Block elimination of the band matrix the reference builds (bead 1 uncoupled to bead 2),
    all chains at once from their last beads, shorter chains joining as they end; the lowest
    eigenvalue by subspace iteration through the factors, shifted once below it."""
    sp, ns, betan, chains = _ring_inputs(case, seed)
    C, N, D, nv = len(ns), max(ns), sp.ndof, 8
    eye = torch.eye(D, dtype=torch.float64, device=DEV)
    c = torch.tensor([1.0 / bn ** 2 for bn in betan], dtype=torch.float64, device=DEV)
    H = eye.repeat(C, N, 1, 1)  # bead j of chain k sits at slot N - n_k + j; unit blocks before
    on = torch.zeros(N, C, dtype=torch.bool, device=DEV)  # coupled to the slot before it
    real = torch.zeros(N, C, dtype=torch.bool, device=DEV)
    for k, (n, x) in enumerate(zip(ns, chains)):
        H[k, N - n:] = _evb_hessian(sp, torch.as_tensor(x, device=DEV)) + 2.0 * c[k] * eye
        real[N - n:, k] = True
        on[N - n + 2:, k] = True
    H = H.transpose(0, 1).contiguous()
    real_f, on_c = real.to(torch.float64), on * c

    def factor(sigma):
        S, ld, prev = [], torch.zeros(C, dtype=torch.float64, device=DEV), None
        for j in range(N):
            A = H[j] - (sigma * real_f[j])[:, None, None] * eye
            if prev is not None:
                A = A - (on_c[j] ** 2)[:, None, None] * prev
            L = torch.linalg.cholesky_ex(A)[0]
            ld += real_f[j] * 2.0 * torch.log(torch.diagonal(L, dim1=1, dim2=2)).sum(1)
            prev = torch.cholesky_inverse(L)
            S.append(prev)
        return S, ld

    def solve(S, v):  # v (N, C, D, nv)
        t = [None] * N
        for j in range(N):
            z = v[j] if j == 0 else v[j] + on_c[j][:, None, None] * t[j - 1]
            t[j] = torch.bmm(S[j], z)
        for j in range(N - 2, -1, -1):
            t[j] = t[j] + on_c[j + 1][:, None, None] * torch.bmm(S[j], t[j + 1])
        return torch.stack(t) * real_f[:, :, None, None]

    def iterate(S, v, sigma, its):
        for _ in range(its):
            w = solve(S, v)
            u = w.transpose(0, 1).reshape(C, N * D, nv)
            u = torch.linalg.qr(u)[0]
            v = u.reshape(C, N, D, nv).transpose(0, 1).contiguous()
            w = solve(S, v).transpose(0, 1).reshape(C, N * D, nv)
            B = torch.bmm(u.transpose(1, 2).contiguous(), w)
            th, R = torch.linalg.eigh(0.5 * (B + B.transpose(1, 2)))
            v = torch.bmm(w, R.contiguous()).reshape(C, N, D, nv).transpose(0, 1).contiguous()
        return v, sigma + 1.0 / th[:, -1]

    zero = torch.zeros(C, dtype=torch.float64, device=DEV)
    S, ld = factor(zero)
    v = torch.randn(N, C, D, nv, dtype=torch.float64, device=DEV,
                    generator=torch.Generator(DEV).manual_seed(1)) * real_f[:, :, None, None]
    v, eta = iterate(S, v, zero, 12)
    sigma = 0.97 * eta  # below eta_1: the Ritz value bounds it from above, within 1 per cent by now
    S, _ = factor(sigma)
    v, eta = iterate(S, v, sigma, 16)
    return dict(logdet=ld - torch.log(eta), nneg=torch.zeros(C, dtype=torch.int32, device=DEV), eta=eta)


def exact(case, seed):
    if case["path"] == "batch":
        return _exact_batch(case, seed)
    if case["path"] == "chain":
        return _exact_chain(case, seed)
    if case["path"] in ("action", "hvp"):
        return _exact_action(case, seed)
    if case["path"] == "logdet":
        return _exact_logdet(case, seed)
    return None  # iterates of a capped search: no value apart from the method's
