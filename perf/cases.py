"""Performance cases of the MD-step solver: what a user's program has it do, through softmold_amd.

Kinds (each through the public Python API):

- md:       one stretch of a simulation between two stored frames: Solver.run of `steps` steps
            from the state the last pass left, then Solver.download of the whole state (what
            md_hip does between two store events).  `graph` replays captured 8-step blocks,
            as the autotuner chooses for some systems; `replicas` > 1 is a sweep of uneven
            vesicles stepped as one batch (softmold_amd.sweep).
- frames:   a frame of a stored trajectory evaluated: upload, forces, energies.
- energies: FP64 energies and the dU of a trial box change at the resident state (what a
            Monte-Carlo driver or a measurement loop asks for).
- fit:      one objective and gradient of a constant-fitting loop (softmold_amd.adjoint).
- response: one block of the fluctuation-formula sampler over independent copies
            (softmold_amd.response.sample): steps, box, energies, dU/dtheta.
- radius:   the vesicle radius of a sweep's replicas, read after every stored frame.

Systems are the generators' vesicles and bilayers at areal density 3.45 with thermal
displacements, so cells hold the uneven numbers of beads they hold in a running simulation.
Velocities, accelerations and forces are held in 32 bits by the solver and are returned as
such; positions, boxes and energies are 64-bit.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from softmold_amd import Mpd, Solver, adjoint, response

DENSITY = 3.45
TAIL = 3
JITTER = 0.1      # thermal displacement of a bead, of the order of a bond's at k = 100, T = 3


def _md(name, model, lipids, steps=16, delta=0.0, tension=0.0, graph=False):
    return {"name": name, "kind": "md", "model": model, "lipids": lipids, "replicas": 1, "steps": steps,
            "delta": delta, "tension": tension, "graph": graph}


def listed():
    return [
        # the smallest vesicle that the tests and the smoke run step: latency and launches
        _md("md vesicle 500", "vesicle", 500),
        # the 5000-lipid vesicle of the known answers: an ordinary small run
        _md("md vesicle 5000", "vesicle", 5000),
        # a small bilayer under box moves, stepped in captured 8-step blocks
        _md("md bilayer 4000 graph", "bilayer", 4000, delta=0.01, graph=True),
        # the vesicle that the benchmark is quoted on
        _md("md vesicle 80000", "vesicle", 80000, steps=24),
        # the largest bilayer of the generator, with its box moves
        _md("md bilayer 1000000", "bilayer", 1000000, steps=24, delta=0.01),
        # the tension x temperature sweep: 64 uneven vesicles stepped as one batch
        {"name": "md sweep 64", "kind": "md", "model": "vesicle", "lipids": 40000, "replicas": 64, "steps": 24,
         "delta": 0.01, "tension": 1.0, "graph": False},
        # analysis of stored frames of an odd-sized vesicle
        {"name": "frames vesicle 12347", "kind": "frames", "model": "vesicle", "lipids": 12347},
        # measurements and trial box changes of a mid-sized bilayer and of the benchmark's vesicle
        {"name": "energies bilayer 30011", "kind": "energies", "model": "bilayer", "lipids": 30011},
        {"name": "energies vesicle 80000", "kind": "energies", "model": "vesicle", "lipids": 80000},
        # one gradient of the fitting loop on the 4000-lipid bilayer
        {"name": "fit bilayer 4000", "kind": "fit", "model": "bilayer", "lipids": 4000, "steps": 24, "checkpoint": 6},
        # one sampling block of the response estimator: 64 copies of the 400-lipid bilayer
        {"name": "response bilayer 64x400", "kind": "response", "model": "bilayer", "lipids": 400, "replicas": 64,
         "steps": 16, "delta": 0.05},
        # the radii of a small sweep
        {"name": "radius 16x2000", "kind": "radius", "model": "vesicle", "lipids": 2000, "replicas": 16},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["md", "md", "md", "sweep", "frames", "energies", "fit", "response", "radius"])
    model = rng.choice(["vesicle", "bilayer"])
    if kind == "md":
        lipids = _log_int(rng, 300, 200000 if model == "vesicle" else 500000)
        return {"kind": "md", "model": model, "lipids": lipids, "replicas": 1, "steps": 8 * rng.randint(1, 3),
                "delta": rng.choice([0.0, 0.01]) if model == "vesicle" else rng.choice([0.01, 0.05]),
                "tension": rng.choice([0.0, 0.5]), "graph": rng.random() < 0.3}
    if kind == "sweep":
        return {"kind": "md", "model": "vesicle", "lipids": _log_int(rng, 3000, 20000), "replicas": rng.randint(2, 48),
                "steps": 8 * rng.randint(1, 3), "delta": 0.01, "tension": 1.0, "graph": rng.random() < 0.3}
    if kind == "frames":
        return {"kind": "frames", "model": model, "lipids": _log_int(rng, 300, 100000)}
    if kind == "energies":
        return {"kind": "energies", "model": model, "lipids": _log_int(rng, 300, 200000)}
    if kind == "fit":
        return {"kind": "fit", "model": "bilayer", "lipids": _log_int(rng, 300, 6000), "steps": rng.randint(8, 24),
                "checkpoint": rng.randint(3, 8)}
    if kind == "response":
        return {"kind": "response", "model": "bilayer", "lipids": _log_int(rng, 300, 2000), "replicas": rng.randint(8, 64),
                "steps": 8 * rng.randint(1, 2), "delta": 0.05}
    return {"kind": "radius", "model": "vesicle", "lipids": _log_int(rng, 300, 20000), "replicas": rng.randint(1, 24)}


# ---- systems ----------------------------------------------------------------------------
def _system(case, lipids, seed):
    """A generator system with thermally displaced beads."""
    generate = Mpd.liposome if case["model"] == "vesicle" else Mpd.bilayer
    m = generate(seed % (1 << 30), lipids, DENSITY)
    d = m.system()
    m.close()
    rng = np.random.default_rng(seed)
    box = np.asarray(d["box"])
    p = d["pos"] + rng.normal(0.0, JITTER, d["pos"].shape)
    p = np.where(p >= box, p - box, np.where(p < 0.0, p + box, p))
    d["pos"] = np.clip(p, 0.0, box)
    d["seed"] = int(seed)
    d["delta_lxy"] = case.get("delta", 0.0)
    d["tension"] = case.get("tension", 0.0)
    return d


def _systems(case, seed):
    R = case.get("replicas", 1)
    if R == 1:
        return [_system(case, case["lipids"], seed)]
    rng = np.random.default_rng([case["lipids"], R])   # the counts are the sweep's, whatever the seed
    hi = case["lipids"]
    side = int(math.ceil(math.sqrt(R)))
    out = []
    for r in range(R):
        same = case["kind"] != "md"   # a sweep's vesicles are uneven, the copies of the samplers alike
        n = hi if same else int(round(math.exp(rng.uniform(math.log(hi / 20), math.log(hi)))))
        d = _system(case, n, seed + 1000 * (r + 1))
        if not same:
            d["tension"] = case["tension"] * (r % side) / max(1, side - 1)
            d["temperature"] *= 0.9 + 0.2 * ((r // side) % side) / max(1, side - 1)
        out.append(d)
    return out


def prepare(case, seed):
    kind = case["kind"]
    systems = _systems(case, seed)
    solver = Solver.batch(systems) if len(systems) > 1 else Solver.from_system(systems[0])
    state = {"case": case, "solver": solver}
    if kind == "md":
        if case["graph"]:
            solver.tune("graph", 1)
        solver.init_forces()
        state["step"] = 1
    elif kind == "frames":
        state["frame"] = _frame(systems[0], seed)
    elif kind == "energies":
        state["scale"] = _scale(seed)
    elif kind == "fit":
        solver.init_forces()
        state["theta"] = _theta(seed)
    elif kind == "response":
        solver.init_forces()
        state["step"] = 1
    return state


def _frame(d, seed):
    """The next frame of the trajectory: every bead a little further."""
    p = d["pos"] + np.random.default_rng([seed, 1]).normal(0.0, 0.02, d["pos"].shape)
    return np.clip(p, 0.0, np.asarray(d["box"]))


def _scale(seed):
    """A volume-conserving trial scaling of the size a box move proposes."""
    f = 1.0 + 1e-4 * np.random.default_rng([seed, 2]).uniform(-1.0, 1.0)
    return np.array([f, f, 1.0 / (f * f)])


def _theta(seed):
    """Umin, Umax of the tail-tail rows, k_bond and k_bend, around the generators' values."""
    return np.array([-6.0, 200.0, 100.0, 100.0]) * (1.0 + 0.02 * np.random.default_rng([seed, 3]).uniform(-1.0, 1.0, 4))


def run(state):
    case, s = state["case"], state["solver"]
    kind = case["kind"]
    if kind == "md":
        s.run(state["step"], case["steps"])
        state["step"] += case["steps"]
        pos, vel, acc, box = s.download()
        return {"pos": pos, "vel": vel.astype(np.float32), "acc": acc.astype(np.float32), "box": box}
    if kind == "frames":
        s.upload(pos=state["frame"])
        fp, fc = s.compute_forces()
        return {"pair": fp.astype(np.float32), "chain": fc.astype(np.float32), "energies": s.measure()}
    if kind == "energies":
        u = s.measure()
        du = s.potential_delta(state["scale"])
        return {"energies": u, "delta": np.asarray(du)}
    if kind == "fit":
        adjoint.set_params(s, (TAIL, TAIL), state["theta"])
        J, g = adjoint.objective(s, (TAIL, TAIL), case["steps"], case["checkpoint"])
        return {"J": J, "grad": g}
    if kind == "response":
        out = response.sample(s, (TAIL, TAIL), state["step"], case["steps"], case["steps"], case["lipids"])
        state["step"] += case["steps"]
        return out
    return {"radius": np.atleast_1d(s.vesicle_radius())}


def work(case):
    """Bytes: per bead and step the position (24), velocity (12) and acceleration (12) read and
    written once, the forces stay in the step.  Flops: each unordered pair within the cutoff
    once (about 27 a bead: 9 for the distance, 14 for the force, 6 to add it to both), the
    chain terms (about 120) and the noise and kicks (about 60)."""
    kind = case["kind"]
    R = case.get("replicas", 1)
    mean = (1.0 - 1.0 / 20) / math.log(20.0) if kind == "md" and R > 1 else 1.0   # of exp(U[ln hi/20, ln hi]) / hi
    n = 3.0 * case["lipids"] * R * mean
    pair, step_b, step_f = 27 * 29.0, 96.0, 27 * 29.0 + 180.0
    if kind == "md":
        return {"bytes": n * step_b * case["steps"], "flops": n * step_f * case["steps"]}
    if kind == "frames":
        return {"bytes": n * (24 + 24 + 12), "flops": n * (2 * pair + 240)}
    if kind == "energies":
        return {"bytes": n * (2 * 24 + 12), "flops": n * (3 * pair + 360)}
    if kind == "fit":   # forward and energies, the recomputed forward, the Hessian-vector products
        k = case["steps"]
        return {"bytes": n * k * (2 * step_b + 24 + 8 * 24), "flops": n * k * (2 * step_f + pair + 3 * pair)}
    if kind == "response":
        return {"bytes": n * (step_b * case["steps"] + 4 * 24), "flops": n * (step_f * case["steps"] + 3 * pair + 360)}
    return {"bytes": n / 3 * 24, "flops": n / 3 * 20}


# ---- the same in plain torch, 64 bits ------------------------------------------------------
def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


class _Ref:
    """One system in 64-bit torch: pair and chain forces, energies, the Langevin step and the
    box move.  The noise is Philox4x32-10 keyed by (seed, step, bead)."""

    SLICE = 1 << 25   # candidate pairs looked at together

    def __init__(self, d, theta=None):
        dev = self.dev = _dev()
        f8 = lambda a: torch.as_tensor(np.asarray(a, np.float64), device=dev)
        self.x, self.v = f8(d["pos"]).clone(), f8(d["vel"]).clone()
        self.type = torch.as_tensor(d["type"], device=dev).long()
        self.box = f8(d["box"]).clone()
        self.nt, self.rc, self.dt = d["n_types"], float(d["cutoff"]), float(d["dt"])
        self.F, self.U = f8(d["fconst"]).reshape(-1, 6), f8(d["uconst"]).reshape(-1, 6)
        self.gamma, self.T, self.seed = float(d["gamma"]), float(d["temperature"]), int(d["seed"])
        self.sigma = math.sqrt(6.0 * self.T * self.gamma / self.dt)
        self.delta, self.tension = float(d["delta_lxy"]), float(d["tension"])
        (start, count, length), (self.l0, self.kb, self.c0, self.kt) = d["chain"][0], d["chain_const"][0]
        self.p0 = torch.arange(int(count), device=dev) * int(length) + int(start)
        assert length == 3
        if theta is not None:
            umin, umax, self.kb, self.kt = theta[0], theta[1], theta[2], theta[3]
            row = TAIL * self.nt + TAIL
            rm, rc = self.F[row, 0], self.F[row, 3]
            w = rc - rm
            z = torch.zeros((), dtype=torch.float64, device=dev)
            fr = torch.stack([rm, 2 * (umax - umin) / rm**2, z, rc, 6 * umin / w**2, 6 * umin / w**3])
            ur = torch.stack([rm, (umax - umin) / rm**2, umin + z, rc, 3 * umin / w**2, 2 * umin / w**3])
            put = lambda T, r: torch.cat([T[:row], r[None], T[row + 1:]])
            self.F, self.U = put(self.F, fr), put(self.U, ur)

    def image(self, d):
        L = self.box
        return d - L * (d > L / 2).double() + L * (d < -L / 2).double()

    @torch.no_grad()
    def pairs(self, x, margin=0.0):
        """Index pairs (i, j), each once, closer than the cutoff plus margin."""
        n, dev, rc = len(x), self.dev, self.rc
        nc = (self.box / rc).long()
        c = torch.minimum((x / (self.box / nc)).long(), nc - 1).clamp_(min=0)
        key = c[:, 0] + nc[0] * (c[:, 1] + nc[1] * c[:, 2])
        skey, order = torch.sort(key, stable=True)
        uk, cnt = torch.unique_consecutive(skey, return_counts=True)
        first = torch.cumsum(cnt, 0) - cnt
        sc, sx = c[order], x[order]
        shell = [(0, 0, 0), (1, 0, 0), (0, 1, 0), (1, 1, 0), (0, 0, 1), (1, 0, 1), (0, 1, 1), (1, 1, 1),
                 (-1, 0, 1), (0, -1, 1), (-1, 1, 1), (1, -1, 1), (-1, -1, 1), (1, -1, 0)]
        I, J = [], []
        step = max(1, min(n, self.SLICE // 64))
        for dx in shell:
            nb = (sc + torch.tensor(dx, device=dev)) % nc
            nk = nb[:, 0] + nc[0] * (nb[:, 1] + nc[1] * nb[:, 2])
            at = torch.searchsorted(uk, nk).clamp_(max=len(uk) - 1)
            m = torch.where(uk[at] == nk, cnt[at], 0)
            f = first[at]
            for a in range(0, n, step):
                mm = m[a:a + step]
                i = torch.repeat_interleave(torch.arange(a, min(n, a + step), device=dev), mm)
                j = torch.arange(len(i), device=dev) - torch.repeat_interleave(torch.cumsum(mm, 0) - mm, mm)
                j += torch.repeat_interleave(f[a:a + step], mm)
                keep = self.image(sx[i] - sx[j]).square().sum(1) < (rc + margin) ** 2
                if dx == (0, 0, 0):
                    keep &= i < j
                I.append(order[i[keep]])
                J.append(order[j[keep]])
        return torch.cat(I), torch.cat(J)

    def force(self, x):
        """(pair, chain) forces; differentiable in x and theta."""
        f = torch.zeros_like(x)
        i, j = self.pairs(x)
        for a in range(0, len(i), self.SLICE):
            ii, jj = i[a:a + self.SLICE], j[a:a + self.SLICE]
            d = self.image(x[ii] - x[jj])
            r = d.square().sum(1).sqrt()
            C = self.F[self.type[ii] * self.nt + self.type[jj]]
            inner = r < C[:, 0]
            m = torch.where(inner, C[:, 0] - r, C[:, 3] - r)
            mag = torch.where(inner, (C[:, 1] - C[:, 2] * m) * m, (C[:, 4] - C[:, 5] * m) * m) / r
            mag = torch.where(r < self.rc, mag, torch.zeros_like(mag))
            fd = d * mag[:, None]
            f = f.index_add(0, ii, fd).index_add(0, jj, -fd)
        p = self.p0
        da, db = self.image(x[p] - x[p + 1]), self.image(x[p + 1] - x[p + 2])
        ra, rb = da.norm(dim=1, keepdim=True), db.norm(dim=1, keepdim=True)
        fa, fb = -(ra - self.l0) * self.kb / ra * da, -(rb - self.l0) * self.kb / rb * db
        ua, ub = da / ra, db / rb
        cos = (ua * ub).sum(1, keepdim=True)
        mag = (self.c0 - cos) * self.kt
        A, B = mag / ra * (ub - ua * cos), mag / rb * (ua - ub * cos)
        c = torch.zeros_like(x).index_add(0, p, fa + A).index_add(0, p + 1, fb - fa + B - A).index_add(0, p + 2, -fb - B)
        return f, c

    def pair_u(self, r, C):
        a, b = C[:, 0] - r, C[:, 3] - r
        u = torch.where(r <= C[:, 0], C[:, 1] * a * a + C[:, 2], b * b * (C[:, 4] - b * C[:, 5]))
        return torch.where(r < self.rc, u, torch.zeros_like(u))

    def chain_u(self, da, db):
        ra, rb = da.norm(dim=1), db.norm(dim=1)
        cos = (da * db).sum(1) / (ra * rb)
        bond = (0.5 * self.kb * ((ra - self.l0) ** 2 + (rb - self.l0) ** 2)).sum()
        return bond, (0.5 * self.kt * (self.c0 - cos) ** 2).sum()

    def energies(self, x, scale=None):
        """(U_pair, U_chain), or U(old) - U(scaled) of both."""
        i, j = self.pairs(x, 0.01 if scale is not None else 0.0)
        up = torch.zeros((), dtype=torch.float64, device=self.dev)
        for a in range(0, len(i), self.SLICE):
            ii, jj = i[a:a + self.SLICE], j[a:a + self.SLICE]
            d = self.image(x[ii] - x[jj])
            C = self.U[self.type[ii] * self.nt + self.type[jj]]
            u = self.pair_u(d.square().sum(1).sqrt(), C)
            if scale is not None:
                u = u - self.pair_u((d * scale).square().sum(1).sqrt(), C)
            up = up + u.sum()
        p = self.p0
        da, db = self.image(x[p] - x[p + 1]), self.image(x[p + 1] - x[p + 2])
        uc = sum(self.chain_u(da, db))
        if scale is not None:
            uc = uc - sum(self.chain_u(da * scale, db * scale))
        return up, uc

    @torch.no_grad()
    def du_dtheta(self, x):
        """dU/d(Umin, Umax of the tail-tail rows, k_bond, k_bend)."""
        i, j = self.pairs(x)
        tt = (self.type[i] == TAIL) & (self.type[j] == TAIL)
        r = self.image(x[i[tt]] - x[j[tt]]).norm(dim=1)
        rm, _, _, rc = [float(c) for c in self.U[TAIL * self.nt + TAIL][:4]]
        w, a, b = rc - rm, (rm - r) / rm, rc - r
        inn, out = r <= rm, (r > rm) & (r < self.rc)
        dmin = torch.where(inn, 1.0 - a * a, b * b * (3.0 / w**2 - 2.0 * b / w**3) * out.double()).sum()
        dmax = (a * a * inn.double()).sum()
        p = self.p0
        bond, bend = self.chain_u(self.image(x[p] - x[p + 1]), self.image(x[p + 1] - x[p + 2]))
        return torch.stack([dmin, dmax, bond / self.kb, bend / self.kt])

    def philox(self, c0, step, tag):
        M = 0xFFFFFFFF
        n = len(c0)
        full = lambda w: torch.full((n,), w & M, dtype=torch.int64, device=self.dev)
        c = [c0, full(step), full(step >> 32), full(tag)]
        k0, k1 = self.seed & M, (self.seed >> 32) & M

        def mul(a, m):   # 32 x 32 -> (hi, lo) without leaving int64
            al, ah, ml, mh = a & 0xFFFF, a >> 16, m & 0xFFFF, m >> 16
            ll, lh, hl, hh = al * ml, al * mh, ah * ml, ah * mh
            mid = (ll >> 16) + (lh & 0xFFFF) + (hl & 0xFFFF)
            return hh + (lh >> 16) + (hl >> 16) + (mid >> 16), ((mid & 0xFFFF) << 16) | (ll & 0xFFFF)

        for _ in range(10):
            h0, l0 = mul(c[0], 0xD2511F53)
            h1, l1 = mul(c[2], 0xCD9E8D57)
            c = [h1 ^ c[1] ^ k0, l1, h0 ^ c[3] ^ k1, l0]
            k0, k1 = (k0 + 0x9E3779B9) & M, (k1 + 0xBB67AE85) & M
        return c

    @staticmethod
    def psi(w):
        return ((w >> 8).double() / 8388608.0 - 1.0) + 1.0 / 16777216.0

    def accel(self, x, v, step, tag):
        f, c = self.force(x)
        w = self.philox(torch.arange(len(x), device=self.dev), step, tag)
        xi = torch.stack([self.psi(w[0]), self.psi(w[1]), self.psi(w[2])], 1)
        return f + c - self.gamma * v + self.sigma * xi

    def begin(self):
        self.a = self.accel(self.x, self.v, 0, 2)

    def step(self, s, sample=None):
        """Step s; returns U_pair + U_chain after the kick when asked (before the box move)."""
        h = 0.5 * self.dt
        v = self.v + self.a * h
        x = self.x + v * self.dt
        L = self.box
        x = x - L * (x > L).double()
        x = x + L * (x < 0).double()
        self.a = self.accel(x, v, s, 0)
        self.v, self.x = v + self.a * h, x
        u = sum(self.energies(x)) if sample else None
        if s % 8 == 0 and self.delta != 0.0:
            self.move(s)
        return u

    def move(self, s):
        w = self.philox(torch.zeros(1, dtype=torch.int64, device=self.dev), s, 1)
        f = self.delta * float(self.psi(w[0]))
        u = ((int(w[1]) >> 5) * 67108864.0 + (int(w[2]) >> 6)) / 9007199254740992.0
        Lx, Ly, Lz = (float(q) for q in self.box)
        new = torch.tensor([Lx + f, Ly + f, Lz * (Lx * Ly) / ((Lx + f) * (Ly + f))], dtype=torch.float64, device=self.dev)
        scale = new / self.box
        dp = float(sum(self.energies(self.x, scale))) + self.tension * ((Lx + f) * (Ly + f) - Lx * Ly)
        if dp >= 0.0 or math.exp(dp / self.T) >= u:
            self.x, self.box = self.x * scale, new


def _cat(parts):
    return np.concatenate([t.detach().cpu().numpy() for t in parts])


def exact(case, seed):
    kind = case["kind"]
    if kind == "fit":
        return _exact_fit(case, seed)
    with torch.no_grad():
        if kind == "md":
            if work(case)["flops"] > 8e10:   # the largest take longer than it is worth
                return None
            refs = [_Ref(d) for d in _systems(case, seed)]
            for q in refs:
                q.begin()
                for s in range(1, case["steps"] + 1):
                    q.step(s)
            box = np.stack([q.box.cpu().numpy() for q in refs])
            return {"pos": _cat(q.x for q in refs), "vel": _cat(q.v for q in refs), "acc": _cat(q.a for q in refs),
                    "box": box[0] if len(refs) == 1 else box}
        if kind == "frames":
            d = _systems(case, seed)[0]
            q = _Ref(d)
            q.x = torch.as_tensor(_frame(d, seed), device=q.dev)
            f, c = q.force(q.x)
            up, uc = q.energies(q.x)
            return {"pair": f.cpu().numpy(), "chain": c.cpu().numpy(),
                    "energies": np.array([float(up), float(uc), float(0.5 * q.v.square().sum())])}
        if kind == "energies":
            q = _Ref(_systems(case, seed)[0])
            up, uc = q.energies(q.x)
            dp, dc = q.energies(q.x, torch.as_tensor(_scale(seed), device=q.dev))
            return {"energies": np.array([float(up), float(uc), float(0.5 * q.v.square().sum())]),
                    "delta": np.array([float(dp), float(dc)])}
        if kind == "response":
            a, U, D = [], [], []
            for d in _systems(case, seed):
                q = _Ref(d)
                q.begin()
                for s in range(1, case["steps"] + 1):
                    q.step(s)
                a.append(2.0 * float(q.box[0] * q.box[1]) / case["lipids"])
                U.append(float(sum(q.energies(q.x))))
                D.append(q.du_dtheta(q.x).cpu().numpy())
            return {"a": np.array([a]), "U": np.array([U]), "D": np.array([D])}
        out = []
        for d in _systems(case, seed):
            h = d["pos"][d["type"] == 2]
            L, p0 = np.asarray(d["box"]), d["pos"][0]
            t = h - p0
            com = (h - np.where(t > L / 2, L, 0.0) + np.where(t < -L / 2, L, 0.0)).mean(0)
            t = h - com
            t = t + np.where(t > L / 2, L, 0.0) - np.where(t < -L / 2, L, 0.0)
            out.append(np.sqrt((t * t).sum(1)).mean())
        return {"radius": np.array(out)}


def _exact_fit(case, seed):
    d = _systems(case, seed)[0]
    theta = torch.tensor(_theta(seed), dtype=torch.float64, device=_dev(), requires_grad=True)
    q = _Ref(d, theta)
    q.begin()
    J = sum(q.step(s, sample=True) for s in range(1, case["steps"] + 1)) / case["steps"]
    (g,) = torch.autograd.grad(J, theta)
    return {"J": float(J.detach()), "grad": g.detach().cpu().numpy()}
