"""The engine's workloads as timed cases, through the Python binding's entry points.

A case is a dict of plain values; `kind` says which calls a pass makes:

  attempt   one Metropolis attempt through the Action interface: the proposal, its
            kinetic and pair action in both modes, accept
  block     one sweep of every replica with its estimators, then what a block's
            write reads: observables, counters and, with `dump`, the paths
  bosons    permuting bisections (the iterative walk) of every replica
  table     permuting bisections (the cycle table) of every replica
  gradient  dS/dr of every bead (adjoint, or the reference's finite differences)
  measure   every observable of uploaded paths, without moves
  restart   a stored path goes up, rho_k and the energies come back

Sizes are the configurations of simpimc_amd.system, the test suite and bench.py:
12 to 1024 particles, 16 to 200 slices, one chain to hundreds of replicas, odd
sizes among them.  `exact` holds a plain torch restatement of the actions, their
gradients and the estimators in 64 bits.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

from simpimc_amd import abi, system

PAIRS = ("bare", "david", "ilkka")
ENERGIES = {"thermal": abi.ENERGY_THERMAL, "compat": abi.ENERGY_VIRIAL_COMPAT, "adjoint": abi.ENERGY_VIRIAL_ADJOINT}
GR_BINS = 200  # g(r) bins of every workload


def _case(name, kind, pair, n, m, replicas=1, level=3, k_shell=25.5, **more):
    return {"name": name, "kind": kind, "pair": pair, "n": n, "m": m, "replicas": replicas, "level": level,
            "k_shell": k_shell, **more}


def listed():
    return [
        # a drop-in caller that keeps its own Metropolis loop: the smallest calls, bound by launches and copies
        _case("attempt_32x32", "attempt", "bare", 32, 32),
        # the plain method on the small electron gas: one chain, thermal energy, replayed from graphs
        _case("chain_32x32", "block", "bare", 32, 32, energy="thermal", adjoint=False, graph=True, dump=True),
        # the plain method on the large electron gas: one chain, adjoint virial energy
        _case("chain_256x128", "block", "david", 256, 128, level=4, k_shell=97.5, energy="adjoint", adjoint=True,
              graph=False, dump=True),
        # 64 clones of uneven sizes, each on its own box and k-set
        _case("uneven_64rep", "block", "uneven", 128, 64, replicas=64, energy="adjoint", adjoint=True, graph=False,
              dump=True),
        # hundreds of clones of the large electron gas: the throughput workload
        _case("batch_256x128_512rep", "block", "david", 256, 128, replicas=512, level=4, k_shell=97.5, energy="adjoint",
              adjoint=True, graph=False, dump=False),
        # few clones of a very large system (half the slices of bench.py's largest one: a sweep stays near a second)
        _case("large_1024x128_8rep", "block", "david", 1024, 128, replicas=8, level=4, k_shell=153.5, energy="adjoint",
              adjoint=True, graph=False, dump=False),
        # clones with the general-grid pair action and the thermal energy
        _case("ilkka_33x32_24rep", "block", "ilkka", 33, 32, replicas=24, energy="thermal", adjoint=False, graph=False,
              dump=True),
        # Bose statistics: permuting bisections of clones of the large electron gas
        _case("bosons_256x128_256rep", "bosons", "david", 256, 128, replicas=256, level=4, k_shell=97.5, attempts=64),
        # Bose statistics by the cycle table, a smaller system with three-particle cycles
        _case("table_32x32_16rep", "table", "bare", 32, 32, replicas=16, level=3, attempts=64, cycle=3),
        # forces of every bead of one large chain
        _case("gradient_256x128", "gradient", "david", 256, 128, level=4, k_shell=97.5, compat=False),
        # measuring stored paths with the reference's own virial estimator, odd sizes
        _case("measure_77x50_12rep", "measure", "bare", 77, 50, replicas=12, energy="compat"),
        # taking up a stored path of a very large system
        _case("restart_1024x128", "restart", "david", 1024, 128, level=4, k_shell=97.5),
    ]


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _n_k(k_shell: float) -> float:
    """about how many vectors a half space holds within |n|^2 < k_shell"""
    return 2.0 / 3.0 * math.pi * k_shell ** 1.5


def draw(rng: random.Random):
    kind = rng.choice(("attempt", "block", "block", "block", "bosons", "table", "gradient", "measure", "restart"))
    pair = rng.choice(("bare", "david", "david", "ilkka")) if kind not in ("measure", "gradient", "restart", "attempt") \
        else rng.choice(("bare", "david"))
    while True:
        n = _log_int(rng, 12, 700)
        m = _log_int(rng, 16, 200)
        replicas = 1 if kind in ("attempt", "gradient", "restart") else _log_int(rng, 1, 200)
        level = rng.randint(2, min(5, int(math.log2(m))))
        c = {"kind": kind, "pair": pair, "n": n, "m": m, "replicas": replicas, "level": level,
             "k_shell": rng.choice((25.5, 25.5, 61.5, 97.5)) if pair == "david" else 25.5}
        beads, links = n * m, 1 << level
        if kind == "block":
            c["energy"] = rng.choice(("thermal", "adjoint", "adjoint"))
            c["adjoint"] = c["energy"] == "adjoint"
            c["graph"] = rng.random() < 0.3
            c["dump"] = replicas <= 64
            rounds = beads / links + n
            per_round = 40e-6 + replicas * links * (4.0 * n / 30e9 + 32.0 * _n_k(c["k_shell"]) / 4e12)
            # the general-grid tables take several times as long, and the path has to be refreshed in one pass
            ok = rounds * per_round * (4.0 if pair == "ilkka" else 1.0) < 0.25 and replicas * n * n * m < 2e8
        elif kind in ("bosons", "table"):
            c["attempts"] = _log_int(rng, 16, 96)
            if kind == "table":
                c["cycle"] = rng.choice((2, 3))
                ok = n <= (200 if c["cycle"] == 2 else 48) and replicas <= 64
            else:
                ok = True
            ok = ok and replicas * n * n < 2e7 and replicas * beads < 8e6
        elif kind == "measure":
            c["energy"] = rng.choice(("thermal", "compat", "adjoint"))
            ok = replicas * n * beads < (6e6 if c["energy"] == "compat" else 3e7)
        elif kind == "gradient":
            c["compat"] = rng.random() < 0.4
            ok = n * beads < (4e6 if c["compat"] else 2e7)
        else:
            ok = n * beads < 1.5e8
        if ok and replicas * beads * 16 < 4e8:
            return c


# ---------------------------------------------------------------------------
# systems and inputs
# ---------------------------------------------------------------------------
def _systems(case):
    kind, n, m, level = case["pair"], case["n"], case["m"], case["level"]
    if kind == "uneven":  # N in {16..n}, M in {16..m}, r_s in [1, 4], each replica's own box and k-set
        rng = np.random.default_rng(11)
        ns = [k for k in (16, 32, 64, 128) if k <= n]
        ms = [k for k in (16, 32, 64) if k <= m]
        return [system.config_c1(n_part=int(rng.choice(ns)), n_bead=int(rng.choice(ms)), r_s=float(rng.uniform(1.0, 4.0)),
                                 n_level=level) for _ in range(case["replicas"])]
    if kind == "bare":
        s = system.config_c1(n_part=n, n_bead=m, n_level=level)
    elif kind == "ilkka":
        s = system.config_ilkka(n_part=n, n_bead=m, n_level=level)
    else:
        s = system.config_c2(n_part=n, n_bead=m, n_level=level, k_shell=case["k_shell"])
    return [s] * case["replicas"]


def _path(s, seed):
    return system.random_path(s, seed=seed, spread=0.05)


def _paths(systems, seed):
    return [_path(s, 1000 * (seed % 1000003) + 17 * r + 1) for r, s in enumerate(systems)]


def _proposals(s, pos, seed, count=16):
    """bisection-like proposals: a particle, 2^level - 1 slices, their displaced positions"""
    rng = np.random.default_rng(seed + 5)
    width = (1 << s.bisect_n_level) - 1
    out = []
    for _ in range(count):
        p, first = int(rng.integers(s.n_part)), int(rng.integers(s.n_bead))
        at = (first + np.arange(width)) % s.n_bead
        out.append((p, first, pos[:, at, p].T + rng.normal(0.0, 0.05, size=(width, 3))))
    return out


def prepare(case, seed):
    systems = _systems(case)
    kind = case["kind"]
    eng = abi.Engine(systems, seed=1 + seed % 1000003)
    pos = _paths(systems, seed)
    if kind != "restart":
        for r, x in enumerate(pos):
            eng.upload(x, r=r)
    st = {"case": case, "eng": eng, "systems": systems}
    if kind == "attempt":
        st["proposals"], st["next"] = _proposals(systems[0], pos[0], seed), 0
    elif kind in ("block", "measure"):
        eng.obs_configure(energy=ENERGIES[case["energy"]], sk_k_cut=_sk_cut(systems), gr_n_r=GR_BINS)
    elif kind in ("bosons", "table"):
        for r in range(len(systems)):
            eng.perm_configure(case["level"], r=r)
            if kind == "table":
                eng.perm_table_configure(case["cycle"], r=r)
    elif kind == "restart":
        st["pos"] = pos[0]
    return st


def _sk_cut(systems):
    return min(0.95 * float(system.kmag(s.L, s.k_n).max()) for s in systems)


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _read(eng, systems):
    """what a block's write reads of every replica: energies, S(k), g(r)"""
    ids = range(len(systems))
    energy = np.stack([eng.obs_read(abi.OBS_ENERGY, r=r)[0] for r in ids])
    sk = np.concatenate([eng.obs_read(abi.OBS_SK, r=r)[0] for r in ids])
    gr = np.stack([eng.obs_read(abi.OBS_GR, r=r)[0] for r in ids])
    return energy, sk, gr


def run(state):
    case, eng, systems = state["case"], state["eng"], state["systems"]
    kind = case["kind"]
    if kind == "attempt":
        p, first, x = state["proposals"][state["next"] % len(state["proposals"])]
        state["next"] += 1
        m = systems[0].n_bead
        b0 = (first - 1) % m
        b1 = b0 + len(x) + 1
        eng.set_proposal(p, first, x)
        out = [eng.get_action(a, mode, b0, b1, [p], 0) for a in (abi.ACTION_KINETIC, abi.ACTION_PAIR)
               for mode in (abi.MODE_OLD, abi.MODE_NEW)]
        eng.accept()
        return np.array(out)
    if kind == "block":
        which = abi.OBS_ENERGY | abi.OBS_SK | abi.OBS_GR
        flags = abi.SWEEP_ENERGY | abi.SWEEP_SK | abi.SWEEP_GR
        flags |= abi.SWEEP_ADJOINT if case["adjoint"] else 0
        flags |= abi.SWEEP_GRAPH if case["graph"] else 0
        eng.obs_reset(which)
        eng.sweep(1, flags)
        energy, sk, gr = _read(eng, systems)
        ids = range(len(systems))
        moves = np.stack([eng.counters(r) for r in ids]).astype(np.int64)
        out = {"energy": energy, "sk": sk, "gr": gr.astype(np.int64), "moves": moves}
        if case["dump"]:
            out["paths"] = np.concatenate([eng.download(r).reshape(-1) for r in ids])
        return out
    if kind in ("bosons", "table"):
        acc = (eng.perm_bisect if kind == "bosons" else eng.perm_table)(case["attempts"])
        ids = range(len(systems))
        sigma = np.stack([eng.perm(r) for r in ids]).astype(np.int64)
        counts = np.concatenate([np.concatenate([c.astype(np.int64) for c in eng.perm_counters(r)[2:]]) for r in ids])
        out = {"accepted": acc.astype(np.int64), "sigma": sigma, "cycles": counts}
        if len(systems) <= 64:
            out["paths"] = np.concatenate([eng.download(r).reshape(-1) for r in ids])
        return out
    if kind == "gradient":
        if case["compat"]:
            return eng.gradient(abi.GRAD_PAIR_SHORT, compat=True)
        return eng.gradient(abi.GRAD_ALL)
    if kind == "measure":
        which = abi.OBS_ENERGY | abi.OBS_SK | abi.OBS_GR
        eng.obs_reset(which)
        eng.obs_accumulate(which)
        energy, sk, gr = _read(eng, systems)
        return {"energy": energy, "sk": sk, "gr": gr.astype(np.int64)}
    eng.upload(state["pos"])
    return {"rho_k": eng.rho_k(), "dbeta": np.array([eng.d_action_d_beta(a) for a in (abi.ACTION_KINETIC, abi.ACTION_PAIR)]),
            "potential": eng.potential(abi.ACTION_PAIR), "virial": eng.kinetic_virial_energy()}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
LINK_FLOPS = {"bare": 60.0, "uneven": 60.0, "david": 110.0, "ilkka": 120.0}  # geometry, tables and sums of one pair on one link
PHASE_FLOPS = 30.0  # e^{i k.r} of one bead's k-vector, two products, and its sums


def work(case):
    systems = _systems(case)
    flops = nbytes = 0.0
    for s in systems:
        n, m, nk, nb = s.n_part, s.n_bead, s.n_k, 1 << case["level"]
        path, rho, u = 24.0 * n * m, 16.0 * nk * m, LINK_FLOPS[case["pair"]]
        pairs = 0.5 * n * (n - 1) * m
        kind = case["kind"]
        if kind in ("attempt", "bosons", "table"):
            att = 1 if kind == "attempt" else case["attempts"]
            flops += att * (2 * nb * n * u + 2 * (nb - 1) * nk * PHASE_FLOPS)
            nbytes += att * ((nb + 1) * n * 24.0 + 2 * (nb - 1) * nk * 16.0)
        elif kind == "block":
            att, dis = (n * m) >> case["level"], n
            flops += 2 * (att * nb + dis * m) * n * u + 2 * (att * (nb - 1) + dis * m) * nk * PHASE_FLOPS
            nbytes += (att * (nb + 1) + dis * m) * n * 24.0 + 2 * (att * (nb - 1) + dis * m) * nk * 16.0
            flops += 2 * pairs * u + m * nk * (n * PHASE_FLOPS if case["adjoint"] else 8.0)
            nbytes += 2 * path + rho
        elif kind == "gradient":
            flops += (6 if case["compat"] else 2) * 2 * pairs * u + (0 if case["compat"] else m * n * nk * PHASE_FLOPS)
            nbytes += 2 * path + (0 if case["compat"] else rho)
        elif kind == "measure":
            f = {"thermal": 1, "adjoint": 3, "compat": 25}[case["energy"]]
            flops += f * pairs * u + m * nk * 8.0 + (m * n * nk * PHASE_FLOPS if case["energy"] == "adjoint" else 0)
            nbytes += path + rho
        else:
            flops += 2 * pairs * u + m * n * nk * PHASE_FLOPS
            nbytes += path + rho
    return {"bytes": nbytes, "flops": flops}


# ---------------------------------------------------------------------------
# the same values in plain torch, 64 bits
# ---------------------------------------------------------------------------
_DEV = "cuda" if torch.cuda.is_available() else "cpu"


def _t(x):
    return torch.as_tensor(np.ascontiguousarray(x), dtype=torch.float64, device=_DEV)


class _Spline:
    """natural cubic splines y[comp][knot] on the uniform grid x, evaluated like the tables of the pair actions:
    outside the grid the edge interval's polynomial continues"""

    def __init__(self, x, y):
        x, y = np.asarray(x, dtype=np.float64), np.atleast_2d(np.asarray(y, dtype=np.float64))
        n = len(x)
        h = np.diff(x)
        curv = np.zeros_like(y)
        cp, dp = np.zeros(n), np.zeros_like(y)
        for i in range(1, n - 1):
            rhs = 6.0 * ((y[:, i + 1] - y[:, i]) / h[i] - (y[:, i] - y[:, i - 1]) / h[i - 1])
            den = 2.0 * (h[i - 1] + h[i]) - h[i - 1] * cp[i - 1]
            cp[i] = h[i] / den
            dp[:, i] = (rhs - h[i - 1] * dp[:, i - 1]) / den
        for i in range(n - 2, 0, -1):
            curv[:, i] = dp[:, i] - cp[i] * curv[:, i + 1]
        self.c = [_t(v) for v in (y[:, :-1], np.diff(y) / h - h * (2.0 * curv[:, :-1] + curv[:, 1:]) / 6.0,
                                  0.5 * curv[:, :-1], np.diff(curv) / (6.0 * h))]
        self.x = _t(x)
        self.x0, self.ih, self.last = float(x[0]), (n - 1) / float(x[-1] - x[0]), n - 2

    def __call__(self, t, comp):
        i = torch.floor((t.detach() - self.x0) * self.ih).clamp(0, self.last).long()
        d = t - self.x[i]
        a, b, c, e = (v[comp][i] for v in self.c)
        return a + d * (b + d * (c + d * e))


class _Action:
    """the pair action of one system: U, dU/dbeta and V of a link from |r|, |r'|, |s|"""

    def __init__(self, s):
        self.s = s
        if s.pair_type == abi.PAIR_BARE:
            self.long = _Spline(s.bare_r_long, s.bare_v_long_r)
            self.scale, self.coef = s.tau, _t(s.v_long_k)
        else:
            self.u, self.du = _Spline(s.david_grid, s.david_u_kj), _Spline(s.david_grid, s.david_du_kj)
            self.scale, self.coef = 1.0, _t(s.v_long_k) * s.tau
        self.const = s.v_long_k_0 * 0.5 * s.n_part ** 2 * s.n_bead - s.v_long_r_0 * 0.5 * s.n_part * s.n_bead

    def _bare(self, r, rp):
        s = self.s
        a, b = (x.clamp(float(s.bare_r[0]), float(s.bare_r[-1])) for x in (r, rp))
        v = 0.5 / a + 0.5 / b
        a, b = (x.clamp(float(s.bare_r_long[0]), float(s.bare_r_long[-1])) for x in (a, b))
        return v - 0.5 * (self.long(a, 0) + self.long(b, 0))

    def _david(self, tab, r, rp, s2, potential):
        lo, hi = float(self.s.david_grid[0]), float(self.s.david_grid[-1])
        a, b = r.clamp(lo, hi), rp.clamp(lo, hi)
        u = 0.5 * (tab(a, 1) + tab(b, 1))
        if potential:
            u = u + 0.5 * (tab(a, 0) + tab(b, 0))
        q, z2 = 0.5 * (r + rp), (r - rp) ** 2
        off = torch.zeros_like(u)
        for k in range(1, self.s.david_n_order + 1):
            for j in range(k + 1):
                off = off + tab(q, k * (k + 1) // 2 + j + 1) * z2 ** j * s2 ** (k - j)
        return u + torch.where((s2 > 0) & (q < hi), off, torch.zeros_like(off))

    def link(self, r, rp, s2):
        return self.s.tau * self._bare(r, rp) if self.s.pair_type == abi.PAIR_BARE else self._david(self.u, r, rp, s2, False)

    def dbeta(self, r, rp, s2):
        return self._bare(r, rp) if self.s.pair_type == abi.PAIR_BARE else self._david(self.du, r, rp, s2, True)

    def potential(self, r, rp):
        if self.s.pair_type == abi.PAIR_BARE:
            return self._bare(r, rp)
        lo, hi = float(self.s.david_grid[0]), float(self.s.david_grid[-1])
        return 0.5 * (self.u(r.clamp(lo, hi), 0) + self.u(rp.clamp(lo, hi), 0))


def _image(d, L):
    return d - torch.round(d.detach() / L) * L


def _geometry(a0, c0, a1, c1, L):
    """|r|, |r'|, |s|^2 of links a -> c, components first: r the minimum image, r' the image nearest r"""
    r = _image(c0 - a0, L)
    rp = c1 - a1
    rp = rp + torch.round((r - rp).detach() / L) * L
    return (r ** 2).sum(0).sqrt(), (rp ** 2).sum(0).sqrt(), ((r - rp) ** 2).sum(0)


def _slabs(n_pairs, m, most=4_000_000):
    step = max(1, most // max(1, n_pairs))
    return [(b, min(m, b + step)) for b in range(0, m, step)]


def _rho(s, x):
    """rho_k[b][k] of the path x[3][M][N]"""
    k = _t(s.k_n) * (2.0 * math.pi / s.L)
    out = []
    for b in range(x.shape[1]):
        ph = k @ x[:, b, :]
        out.append(torch.complex(torch.cos(ph).sum(1), torch.sin(ph).sum(1)))
    return torch.stack(out)


def _pair_sum(s, x, fn):
    i, j = torch.triu_indices(s.n_part, s.n_part, 1, device=x.device)
    nxt = torch.roll(x, -1, 1)
    tot = 0.0
    for b, e in _slabs(len(i), s.n_bead):
        tot += float(fn(x[:, b:e, i], x[:, b:e, j], nxt[:, b:e, i], nxt[:, b:e, j]).sum())
    return tot


def _dbeta(s, act, x, rho2):
    d = _image(x - torch.roll(x, -1, 1), s.L)
    kin = s.n_part * s.n_bead * 3 / (2.0 * s.tau) - float((d ** 2).sum()) / (4.0 * s.lam * s.tau ** 2)
    pair = _pair_sum(s, x, lambda a0, c0, a1, c1: act.dbeta(*_geometry(a0, c0, a1, c1, s.L)))
    return kin, pair + float((rho2.sum(0) * _t(s.v_long_k)).sum()) + act.const


def _potential(s, act, x, rho2):
    def v(a0, c0, a1, c1):
        return act.potential(*((_image(p - q, s.L) ** 2).sum(0).sqrt() for p, q in ((a0, c0), (a1, c1))))

    return _pair_sum(s, x, v) + float((rho2.sum(0) * _t(s.v_long_k)).sum()) + act.const


def _virial_kinetic(s, x):
    step = _image(torch.roll(x, -1, 1) - x, s.L)
    whole = step.sum(1, keepdim=True)  # the window is the whole path
    w = s.n_bead * s.tau
    return s.n_part * s.n_bead * 3 / (2.0 * s.tau) / s.n_bead - float((whole * step).sum()) / (4.0 * s.lam * s.tau) / w


def _adjoint(s, act, x, kinetic):
    """dS/dr[3][M][N] by differentiating the action"""
    x = x.detach().clone().requires_grad_(True)
    i, j = torch.triu_indices(s.n_part, s.n_part, 1, device=x.device)
    for b, e in _slabs(len(i), s.n_bead, 1_000_000):
        at = torch.arange(b, e + 1, device=x.device) % s.n_bead
        y = x[:, at]
        act.link(*_geometry(y[:, :-1, i], y[:, :-1, j], y[:, 1:, i], y[:, 1:, j], s.L)).sum().backward()
    k = _t(s.k_n) * (2.0 * math.pi / s.L)
    for b in range(s.n_bead):
        ph = k @ x[:, b, :]
        (act.scale * act.coef * (torch.cos(ph).sum(1) ** 2 + torch.sin(ph).sum(1) ** 2)).sum().backward()
    if kinetic:
        d = _image(x - torch.roll(x, -1, 1), s.L)
        ((d ** 2).sum() / (4.0 * s.lam * s.tau)).backward()
    return x.grad


def _differences(s, act, x, eps=1e-4):
    """the reference's pair gradient: central differences of the links (b, b + 1) and (b, b - 1) in bead b"""
    n, g = s.n_part, torch.zeros_like(x)
    other = ~torch.eye(n, dtype=torch.bool, device=x.device)
    for b in range(s.n_bead):
        a0, c0 = x[:, b, :, None], x[:, b, None, :]
        for t in ((b + 1) % s.n_bead, (b - 1) % s.n_bead):
            a1, c1 = x[:, t, :, None], x[:, t, None, :]
            for d in range(3):
                f = []
                for sign in (1.0, -1.0):
                    y = a0.clone()
                    y[d] = a0[d] + sign * eps
                    f.append(act.link(*_geometry(y, c0, a1, c1, s.L)))
                g[d, b] += torch.where(other, f[0] - f[1], torch.zeros_like(f[0])).sum(1) / (2.0 * eps)
    return g


def _exact_measure(case, s, act, x):
    rho = _rho(s, x)
    rho2 = rho.real ** 2 + rho.imag ** 2
    kin, pair = _dbeta(s, act, x, rho2)
    if case["energy"] != "thermal":
        g = _differences(s, act, x) if case["energy"] == "compat" else _adjoint(s, act, x, False)
        kin = _virial_kinetic(s, x) + float((g * _image(x - x[:, :1], s.L)).sum()) / (2.0 * s.tau)
    sk = torch.where(_t(system.kmag(s.L, s.k_n)) < _sk_cut([s]), rho2.sum(0), torch.zeros_like(rho2[0]))
    return [kin, pair], sk.cpu().numpy()


def exact(case, seed):
    kind, pair = case["kind"], case["pair"]
    # what the engine's own random numbers decide has no value without its code
    if kind in ("block", "bosons", "table") or pair not in ("bare", "david"):
        return None
    systems = _systems(case)
    s = systems[0]
    act, pos = _Action(s), _paths(systems, seed)
    x = _t(pos[0])
    n, m = s.n_part, s.n_bead
    if kind == "attempt":
        p, first, new = _proposals(s, pos[0], seed)[0]
        b0 = (first - 1) % m
        y = x.clone()
        y[:, (first + torch.arange(len(new), device=x.device)) % m, p] = _t(new).T
        at = (b0 + torch.arange(len(new) + 2, device=x.device)) % m
        others = torch.tensor([q for q in range(n) if q != p], device=x.device)
        kin, pot = [], []
        for z in (x, y):
            a = z[:, at, p]
            kin.append(float((_image(a[:, :-1] - a[:, 1:], s.L) ** 2).sum()) / (4.0 * s.lam * s.tau))
            c = z[:, at][:, :, others]
            u = act.link(*_geometry(a[:, :-1, None], c[:, :-1], a[:, 1:, None], c[:, 1:], s.L)).sum()
            rho = _rho(s, z[:, at[:-1]])
            pot.append(float(u) + act.scale * float((act.coef * (rho.real ** 2 + rho.imag ** 2)).sum()))
        return np.array(kin + pot)
    if kind == "gradient":
        if case["compat"] and n * n * m > 6e6:
            return None
        g = _differences(s, act, x) if case["compat"] else _adjoint(s, act, x, True)
        return g.permute(1, 2, 0).contiguous().cpu().numpy()
    if kind == "measure":
        if len(systems) * n * n * m > 1.2e8 or len(systems) * m > 3000:
            return None
        got = [_exact_measure(case, s, act, _t(p)) for p in pos]
        return {"energy": np.array([e for e, _ in got]), "sk": np.concatenate([k for _, k in got]), "gr": None}
    rho = _rho(s, x)
    rho2 = rho.real ** 2 + rho.imag ** 2
    return {"rho_k": rho.cpu().numpy(), "dbeta": np.array(_dbeta(s, act, x, rho2)), "potential": _potential(s, act, x, rho2),
            "virial": _virial_kinetic(s, x)}
