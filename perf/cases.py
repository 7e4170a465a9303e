"""The work a user of this library has it do, as timed cases.

Eight kinds of case, over the sizes the library is used at: RK4 and MSRK evolutions of one grid
(from the 24^3 long-run problems, where a pass is launches and latency, to the 256^3 binary),
the radiative outer boundary, the right-hand side by itself in each of its forms (fused,
two-pass, INT8-split, block floating point), the constraints, and RK4 steps of the two block
hierarchies. Grids are Brill-Lindquist binaries with seeded smooth perturbations unless a case
says otherwise, steps are dt = h/4.

``exact`` restates the BSSN system, the stencils, the steps and the ghost rules in plain torch
float64, from the equations, without the library.
"""
from __future__ import annotations

import itertools
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "integer-schemes_amd"))

from bssn3d_hip import BSSNEvolution, BSSNSolver, ConstraintSolver, Grid  # noqa: E402
from bssn3d_hip import initial_data as idata  # noqa: E402
from bssn3d_hip.amr import REFINE, AMRHierarchy  # noqa: E402
from bssn3d_hip.patches import config_hierarchy  # noqa: E402

NF = 24
ALPHA, CHI, K, GT, BETA, AT, GTI, BB = 0, 1, 2, 3, 9, 12, 18, 21
# parameters of the evolution (the library's defaults, which every case uses)
ETA, CAHD, SSL_H, SSL_SIG, FLOOR = 2.0, 0.06, 0.6, 20.0, 1e-4
BOX = 16.0                      # extent of the longest axis of the binary grids


# ------------------------------------------------------------------------------- the cases

def _text(n):
    return "x".join(str(v) for v in n)


def _dims(text):
    """[a, b, c] of "axbxc"."""
    return [int(v) for v in text.split("x")]


def _many(text):
    return [_dims(t) for t in text.split(",")]


def listed():
    return [
        # a chunk of a long run between two samples: 24^3 at the production order, ghosts kept as
        # the reference keeps them, then the constraint norms. Launches and latency.
        dict(name="series_24", kind="series", n="24x24x24", order=6, steps=4),
        # the production order at an ordinary size
        dict(name="rk4_128_fd6", kind="rk4", n="128x128x128", order=6, steps=2),
        # the benchmark's workload: the 256^3 binary at order 4
        dict(name="rk4_256_fd4", kind="rk4", n="256x256x256", order=4, steps=2),
        # the multi-step integrator on a ragged grid: start step, then two recurrences
        dict(name="msrk_ragged_fd4", kind="msrk", n="117x90x143", order=4, steps=3),
        # a puncture run in a finite box: radiative ghost zones
        dict(name="radiative_160", kind="radiative", n="160x160x160", order=4, steps=1),
        # the right-hand side alone, as a caller with its own integrator uses it (order 6, ragged)
        dict(name="rhs_fused_ragged_fd6", kind="rhs", scheme="fused", n="121x131x93", order=6),
        # the materialised form, the reference role of the acceptance gate
        dict(name="rhs_twopass_128_fd6", kind="rhs", scheme="twopass", n="128x128x128",
             order=6),
        # derivatives on the INT8 matrix cores
        dict(name="rhs_int8_160", kind="rhs", scheme="int8", n="160x160x160", order=4),
        # the derivative bundle stored in 32-bit block floating point
        dict(name="rhs_bfp32_112", kind="rhs", scheme="bfp32", n="112x112x112", order=4),
        # constraint fields and their norms of a finished run
        dict(name="constraints_144", kind="constraints", n="144x144x144", order=4),
        # nested levels of uneven blocks in one batch, ghosts by the fill program
        dict(name="patches_240", kind="patches", counts="5x5x4,5x4x4,5x4x3",
             cut_seed=0, ghosts="program"),
        # a live octree of 16^3 blocks on three levels
        dict(name="octree_384", kind="octree", roots="4x4x4", refine="4x2x2,6x2x2",
             ghosts="program"),
    ]


def draw(rng):
    def extent(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def box(lo, hi):
        if rng.random() < 0.3:
            return _text([extent(lo, hi)] * 3)
        return _text(extent(lo, hi) for _ in range(3))

    kind = rng.choice(["series", "rk4", "rk4", "rk4", "msrk", "radiative", "rhs", "rhs", "rhs",
                       "constraints", "patches", "octree"])
    if kind == "series":
        return dict(kind=kind, n=_text([rng.randint(12, 48)] * 3), order=rng.choice([4, 6]),
                    steps=rng.randint(1, 6))
    if kind == "rk4":
        order = rng.choice([4, 6, 8])
        return dict(kind=kind, n=box(20, {4: 240, 6: 180, 8: 130}[order]), order=order,
                    steps=rng.randint(1, 2))
    if kind == "msrk":
        return dict(kind=kind, n=box(24, 160), order=rng.choice([4, 6]), steps=rng.randint(2, 3))
    if kind == "radiative":
        return dict(kind=kind, n=box(32, 190), order=rng.choice([4, 6]), steps=1)
    if kind == "rhs":
        scheme = rng.choice(["fused", "fused", "twopass", "int8", "bfp32", "bfp48"])
        return dict(kind=kind, scheme=scheme, n=box(24, 170),
                    order=4 if scheme == "int8" else rng.choice([4, 6]))
    if kind == "constraints":
        return dict(kind=kind, n=box(24, 170), order=rng.choice([4, 6]))
    if kind == "patches":
        counts = _text(rng.randint(4, 5) for _ in range(3)) + ",4x3x3,4x3x3"
        return dict(kind=kind, counts=counts, cut_seed=rng.randint(0, 9999),
                    ghosts=rng.choice(["program", "linked"]))
    return dict(kind=kind, roots=_text([4, rng.randint(3, 4), 4]),
                refine=_text([rng.choice([2, 4]), 2, 2]) + "," +
                _text([rng.choice([2, 4]), rng.choice([2, 4]), 2]),
                ghosts=rng.choice(["program", "linked"]))


# ---------------------------------------------------------------------------- preparation

def _ko_order(order):
    return min(order + 2, 8)


def _binary(n, ng, seed):
    """(grid, state): an equal-mass binary on a box whose longest axis is BOX, the punctures a
    fraction of a cell off the grid planes, 1e-4 perturbations."""
    h = BOX / max(n)
    lo = [-0.5 * v * h for v in n]
    grid = Grid(*n, h, h, h, ng=ng, xmin=lo[0], ymin=lo[1], zmin=lo[2])
    rng = np.random.default_rng(seed)
    off = idata.offgrid_shift(rng, h)
    d = 0.1875 * n[0] * h
    pos = [np.array([-d, 0.0, 0.0]) + off, np.array([d, 0.0, 0.0]) + off]
    return grid, idata.punctures(grid, [0.5, 0.5], pos, amp=1e-4, seed=seed, device="cuda")


def _bump(n, order, seed):
    """(grid, state): flat space on the periodic unit cube, a smooth bump of chi and 1e-8 noise
    (the long-run problems)."""
    grid = Grid.from_domain(tuple(n), order=order)
    amp = 1e-3 * (1.0 + np.random.default_rng(seed).uniform())
    U = idata.robust_stability(grid, amp=1e-8, seed=seed, device="cuda")
    U += idata.hamiltonian_bump(grid, amplitude=amp, device="cuda")
    U -= idata.minkowski(grid, device="cuda")
    return grid, U


def prepare(case, seed):
    kind = case["kind"]
    if kind == "series":
        grid, U = _bump(_dims(case["n"]), case["order"], seed)
        evo = BSSNEvolution(grid, order=case["order"], ko_sigma=0.1, ghosts="carried")
        return dict(case=case, U=U, grid=grid, dt=0.25 * grid.dx, evo=evo,
                    cons=ConstraintSolver(grid, order=case["order"]))
    if kind in ("rk4", "msrk", "radiative"):
        grid, U = _binary(_dims(case["n"]), _ko_order(case["order"]) // 2, seed)
        evo = BSSNEvolution(grid, order=case["order"], ko_sigma=0.1,
                            bc="sommerfeld" if kind == "radiative" else "periodic",
                            integrator="rk4_2_2" if kind == "msrk" else "rk4")
        return dict(case=case, U=U, grid=grid, dt=0.25 * grid.dx, evo=evo)
    if kind == "rhs":
        grid, U = _binary(_dims(case["n"]), _ko_order(case["order"]) // 2, seed)
        return dict(case=case, U=U, grid=grid, dt=0.25 * grid.dx, t=0.5,
                    solver=BSSNSolver(grid, order=case["order"], scheme=case["scheme"]))
    if kind == "constraints":
        grid, U = _binary(_dims(case["n"]), _ko_order(case["order"]) // 2, seed)
        return dict(case=case, U=U, grid=grid,
                    cons=ConstraintSolver(grid, order=case["order"]))
    if kind == "patches":
        H, pos = config_hierarchy(seed=case["cut_seed"], counts=_many(case["counts"]),
                                  device="cuda", hold_punctures=False)
        U = H.empty_pool()
        shift = idata.offgrid_shift(np.random.default_rng(seed), H.boxes[-1].h)
        root = H.boxes[0]
        domain = (H.x0, tuple(root.extent[a] * root.h for a in range(3)))
        for L, box in enumerate(H.boxes):   # one smooth state per level, cut into its blocks
            lo = [H.x0[a] + box.origin[a] * box.h for a in range(3)]
            g = Grid(*box.extent, box.h, box.h, box.h, ng=H.ng, xmin=lo[0], ymin=lo[1],
                     zmin=lo[2])
            F = idata.punctures(g, [0.909, 0.0909], [np.asarray(p) + shift for p in pos],
                                amp=1e-4, seed=seed, device="cuda", domain=domain)
            for b in range(len(H)):
                if H.level[b] == L:
                    H.view(U, b).copy_(F[_patch_slices(H, b)])
        H.sync_(U)
        if case["ghosts"] == "linked":
            H.link, H.linked_program
        return dict(case=case, U=U, H=H, t=0.0, dt=0.25 * H.boxes[-1].h)
    assert kind == "octree"
    roots = _dims(case["roots"])
    H = AMRHierarchy(nb_root=tuple(roots), BS=16, ng=3, levels=3, L=BOX,
                     lo=tuple(-0.5 * BOX * r / roots[0] for r in roots), device="cuda")
    _, F = _binary([16 * r for r in roots], 3, seed)
    U = H.from_global(H.empty_pool(), F)
    at = roots
    for L, r in enumerate(_many(case["refine"])):   # the central r tiles of the level
        lo = [(a - q) // 2 for a, q in zip(at, r)]
        U = H.apply(U, {t: REFINE for t in H.tree.on_level(L)
                        if all(lo[a] <= t[1 + a] < lo[a] + r[a] for a in range(3))})
        at = [2 * a for a in at]
    if case["ghosts"] == "linked":
        H.link, H.linked_program
    return dict(case=case, U=U, H=H, t=0.0, dt=0.25 * H.spacing(H.levels - 1))


def run(state):
    kind = state["case"]["kind"]
    if kind in ("rk4", "msrk", "radiative"):
        return state["evo"].evolve(state["U"], state["dt"], state["case"]["steps"]).data
    if kind == "series":
        out = state["evo"].evolve(state["U"], state["dt"], state["case"]["steps"]).data
        return (out,) + tuple(state["cons"].l2(out))
    if kind == "rhs":
        return state["solver"].rhs(state["U"], t=state["t"], dt=state["dt"]).data
    if kind == "constraints":
        c = state["cons"].constraints(state["U"])
        return (c["H"], c["M0"], c["M1"], c["M2"]) + tuple(state["cons"].l2(state["U"]))
    # the hierarchies step in place, as their run loops do
    state["H"].step_(state["U"], state["t"], state["dt"], ghosts=state["case"]["ghosts"])
    state["t"] += state["dt"]
    return state["U"]


def _patch_slices(H, b):
    """Block b's padded points in its level's padded array."""
    o = H.boxes[H.level[b]].origin
    return (slice(None),) + tuple(
        slice(H.node0[b][a] - o[a], H.node0[b][a] - o[a] + H.layout.S[b][a]) for a in range(3))


# ---------------------------------------------------------------------------- the work

# floating-point operations per point of one right-hand side: 72 first, 33 second and 33 mixed
# derivatives, the algebra (4309), and 24 Kreiss-Oliger terms along three axes
def _rhs_flops(order, ko):
    r, k = order // 2, _ko_order(order) // 2
    stencils = 72 * 4 * r + 33 * (4 * r + 2) + 33 * (2 * r) * (4 * r + 1)
    return stencils + 4309 + (24 * 3 * (4 * k + 2) if ko else 0)


def work(case):
    """Every input read once and every output written once per evaluated step, and the
    operations of its right-hand sides."""
    kind = case["kind"]
    if kind in ("patches", "octree"):
        if kind == "patches":
            H, _ = config_hierarchy(seed=case["cut_seed"],
                                    counts=_many(case["counts"]), device="cpu",
                                    hold_punctures=False)
            pts = sum(int(np.prod(b.n)) for b in H.blocks)
            padded = sum(H.layout.P)
        else:
            nb = int(np.prod(_dims(case["roots"])))
            nb += 8 * sum(int(np.prod(r)) for r in _many(case["refine"]))
            pts, padded = nb * 16 ** 3, nb * 22 ** 3
        return {"bytes": 16 * NF * padded, "flops": 4 * pts * (_rhs_flops(4, True) + 96)}
    pts = int(np.prod(_dims(case["n"])))
    order = case["order"]
    padded = int(np.prod([v + 2 * (_ko_order(order) // 2) for v in _dims(case["n"])]))
    if kind == "rhs":
        return {"bytes": 16 * NF * padded, "flops": padded * _rhs_flops(order, False)}
    if kind == "constraints":
        return {"bytes": (8 * 17 + 8 * 4) * padded, "flops": 2 * padded * 3000}
    evals = 4 * case["steps"] if kind != "msrk" else 1 + 4 + 3 * (case["steps"] - 1)
    out = {"bytes": 16 * NF * padded * case["steps"],
           "flops": evals * pts * (_rhs_flops(order, True) + 96)}
    if kind == "series":
        out["bytes"] += (8 * 17) * padded
        out["flops"] += padded * 3000
    return out


# ---------------------------------------------------------- the same values in plain torch

_D1 = {4: ([8.0, -1.0], 12.0), 6: ([45.0, -9.0, 1.0], 60.0),
       8: ([672.0, -168.0, 32.0, -3.0], 840.0)}
_D2 = {4: ([-30.0, 16.0, -1.0], 12.0), 6: ([-490.0, 270.0, -27.0, 2.0], 180.0),
       8: ([-14350.0, 8064.0, -1008.0, 128.0, -9.0], 5040.0)}
_KO = {6: ([-20.0, 15.0, -6.0, 1.0], 64.0), 8: ([-70.0, 56.0, -28.0, 8.0, -1.0], 256.0)}
_SYM = [[0, 1, 2], [1, 3, 4], [2, 4, 5]]
_PAIRS = [(0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2)]
R3 = range(3)


class _Stencils:
    """Derivatives of the fields of P (24, ..., nx + 2H, ny + 2H, nz + 2H) at its core."""

    def __init__(self, P, H, h, order):
        self.P, self.H, self.h, self.order = P, H, h, order
        self.n = [s - 2 * H for s in P.shape[-3:]]

    def at(self, f, off=(0, 0, 0)):
        H, n = self.H, self.n
        return self.P[f][(Ellipsis,) + tuple(slice(H + off[a], H + off[a] + n[a]) for a in R3)]

    def _shift(self, f, a, k, base=(0, 0, 0)):
        o = list(base)
        o[a] += k
        return self.at(f, o)

    def _first(self, f, a, base=(0, 0, 0)):
        c, _ = _D1[self.order]
        return sum(c[k - 1] * (self._shift(f, a, k, base) - self._shift(f, a, -k, base))
                   for k in range(1, len(c) + 1))

    def d1(self, f, a):
        return self._first(f, a) / (_D1[self.order][1] * self.h)

    def d2(self, f, i, j):
        if i == j:
            c, den = _D2[self.order]
            s = c[0] * self.at(f)
            for k in range(1, len(c)):
                s = s + c[k] * (self._shift(f, i, k) + self._shift(f, i, -k))
            return s / (den * self.h ** 2)
        c, den = _D1[self.order]
        e = [0, 0, 0]
        s = 0.0
        for k in range(1, len(c) + 1):
            for sign in (1, -1):
                e[j] = sign * k
                s = s + sign * c[k - 1] * self._first(f, i, e)
        return s / (den * self.h) ** 2

    def ko(self, f, sigma):
        c, den = _KO[_ko_order(self.order)]
        s = 0.0
        for a in R3:
            s = s + c[0] * self.at(f)
            for k in range(1, len(c)):
                s = s + c[k] * (self._shift(f, a, k) + self._shift(f, a, -k))
        return s * (sigma / (den * self.h))


def _contract(a, b):
    return sum(a[_SYM[i][j]] * b[_SYM[i][j]] for i in R3 for j in R3)


def _inverse(g):
    a = [g[3] * g[5] - g[4] ** 2, g[2] * g[4] - g[1] * g[5], g[1] * g[4] - g[2] * g[3],
         g[0] * g[5] - g[2] ** 2, g[1] * g[2] - g[0] * g[4], g[0] * g[3] - g[1] ** 2]
    det = g[0] * a[0] + g[1] * a[1] + g[2] * a[2]
    return [v / det for v in a], det


class _Geometry:
    """Metric, Christoffels and Ricci tensor of the conformal decomposition at the core."""

    def __init__(self, S):
        s = _SYM
        self.g = g = [S.at(GT + q) for q in range(6)]
        self.ig, _ = _inverse(g)
        ig = self.ig
        self.dg = dg = [[S.d1(GT + q, a) for q in range(6)] for a in R3]
        low = [[0.5 * (dg[j][s[k][i]] + dg[i][s[k][j]] - dg[k][s[i][j]]) for i, j in _PAIRS]
               for k in R3]
        self.C = C = [[sum(ig[s[m][k]] * low[k][q] for k in R3) for q in range(6)] for m in R3]
        self.cal = cal = [_contract(ig, C[m]) for m in R3]
        self.chi = chi = S.at(CHI)
        self.dchi = dchi = [S.d1(CHI, a) for a in R3]
        self.up = up = [sum(ig[s[m][k]] * dchi[k] for k in R3) for m in R3]
        d2c = [S.d2(CHI, i, j) for i, j in _PAIRS]
        lap = _contract(ig, d2c) - 1.5 / chi * sum(dchi[m] * up[m] for m in R3) \
            - sum(cal[m] * dchi[m] for m in R3)
        dG = [[S.d1(GTI + k, a) for a in R3] for k in R3]
        # gl[k][l][m]: Gamma_k with its first lower index raised, gt^lp Gamma_k(p m)
        gl = [[[sum(ig[s[l][p]] * low[k][s[p][m]] for p in R3) for m in R3] for l in R3]
              for k in R3]
        self.R = []
        for q, (i, j) in enumerate(_PAIRS):
            r = -0.5 * _contract(ig, [S.d2(GT + q, a, b) for a, b in _PAIRS])
            for k in R3:
                r = r + 0.5 * (g[s[k][i]] * dG[k][j] + g[s[k][j]] * dG[k][i])
                r = r + 0.5 * cal[k] * (low[i][s[j][k]] + low[j][s[i][k]])
                for m in R3:
                    # gt^lm (Gamma^k_li Gamma_jkm + Gamma^k_lj Gamma_ikm + Gamma^k_im Gamma_klj)
                    r = r + C[k][s[m][i]] * gl[j][m][k] + C[k][s[m][j]] * gl[i][m][k] \
                        + C[k][s[i][m]] * gl[k][m][j]
            c = sum(C[m][q] * dchi[m] for m in R3)
            r = r + 0.5 / chi * (d2c[q] - c + g[q] * lap) - 0.25 / chi ** 2 * dchi[i] * dchi[j]
            self.R.append(r)


def _raised(A, ig):
    s = _SYM
    m = [[sum(ig[s[k][l]] * A[s[l][j]] for l in R3) for j in R3] for k in R3]
    up = [sum(m[i][l] * ig[s[l][j]] for l in R3) for i, j in _PAIRS]
    return m, up, _contract(up, A)


def _rates(P, H, h, dt, t, order, sigma):
    """d/dt of the 24 fields at the core of P (padded by H): right-hand side plus
    Kreiss-Oliger."""
    s = _SYM
    S = _Stencils(P, H, h, order)
    G = _Geometry(S)
    g, ig, C, cal, chi, dchi = G.g, G.ig, G.C, G.cal, G.chi, G.dchi
    b = [S.at(BETA + i) for i in R3]
    al, k0 = S.at(ALPHA), S.at(K)
    A = [S.at(AT + q) for q in range(6)]
    mixA, upA, AA = _raised(A, ig)
    dal = [S.d1(ALPHA, a) for a in R3]
    db = [[S.d1(BETA + i, j) for i in R3] for j in R3]
    div = sum(db[i][i] for i in R3)

    def adv(d):
        return sum(b[a] * d[a] for a in R3)

    out = [None] * NF
    dot = sum(G.up[m] * dal[m] for m in R3)
    DD = []
    for q, (i, j) in enumerate(_PAIRS):
        c = sum(C[m][q] * dal[m] for m in R3) \
            - 0.5 / chi * (dal[i] * dchi[j] + dal[j] * dchi[i] - g[q] * dot)
        DD.append(S.d2(ALPHA, i, j) - c)
    X = [al * G.R[q] - DD[q] for q in range(6)]
    trX = _contract(ig, X) / 3.0
    ham = chi * _contract(ig, G.R) - AA + 2.0 / 3.0 * k0 ** 2
    cahd = CAHD * h * h / (dt * (10.0 * h * h + 1.0))
    sq = torch.sqrt(chi)
    out[ALPHA] = adv(dal) - 2.0 * al * k0 - \
        sq * SSL_H * (al - sq) * math.exp(-0.5 * t * t / SSL_SIG ** 2)
    out[CHI] = adv(dchi) + cahd * chi * ham + 2.0 / 3.0 * chi * (al * k0 - div)
    out[K] = adv([S.d1(K, a) for a in R3]) - chi * _contract(ig, DD) \
        + al * (k0 ** 2 / 3.0 + AA)
    for q, (i, j) in enumerate(_PAIRS):
        lieg = sum(g[s[i][k]] * db[j][k] + g[s[k][j]] * db[i][k] for k in R3)
        lieA = sum(A[s[i][k]] * db[j][k] + A[s[k][j]] * db[i][k] for k in R3)
        AkA = sum(A[s[i][k]] * mixA[k][j] for k in R3)
        out[GT + q] = adv([G.dg[a][q] for a in R3]) + lieg - 2.0 / 3.0 * g[q] * div \
            - 2.0 * al * A[q]
        out[AT + q] = adv([S.d1(AT + q, a) for a in R3]) + chi * (X[q] - g[q] * trX) + lieA \
            - 2.0 / 3.0 * A[q] * div + al * (k0 * A[q] - 2.0 * AkA)
    dK = [S.d1(K, a) for a in R3]
    d2b = [[S.d2(BETA + i, a, c) for a, c in _PAIRS] for i in R3]
    for i in R3:
        r = adv([S.d1(GTI + i, a) for a in R3]) - sum(cal[j] * db[j][i] for j in R3) \
            + 2.0 / 3.0 * cal[i] * div + _contract(ig, d2b[i]) \
            + sum(ig[s[i][j]] * d2b[m][s[j][m]] for j in R3 for m in R3) / 3.0 \
            + 2.0 * al * _contract(C[i], upA) \
            - sum(upA[s[i][j]] * (2.0 * dal[j] + 3.0 * al / chi * dchi[j]) for j in R3) \
            - 4.0 / 3.0 * al * sum(ig[s[i][j]] * dK[j] for j in R3)
        out[GTI + i] = r
        out[BB + i] = r - adv([S.d1(GTI + i, a) for a in R3]) - ETA * S.at(BB + i) \
            + adv([S.d1(BB + i, a) for a in R3])
        out[BETA + i] = 0.75 * S.at(BB + i) + adv([db[j][i] for j in R3])
    if sigma > 0.0:
        out = [out[f] + S.ko(f, sigma) for f in range(NF)]
    return torch.stack(out)


def _constraint_fields(P, H, h, order):
    """Hamiltonian and momentum constraints (4 arrays) at the core of P."""
    s = _SYM
    S = _Stencils(P, H, h, order)
    G = _Geometry(S)
    A = [S.at(AT + q) for q in range(6)]
    _, _, AA = _raised(A, G.ig)
    ham = G.chi * _contract(G.ig, G.R) - AA + 2.0 / 3.0 * S.at(K) ** 2
    dA = [[S.d1(AT + q, a) for q in range(6)] for a in R3]
    out = [ham]
    for i in R3:
        m = -2.0 / 3.0 * S.d1(K, i) - sum(S.at(GTI + j) * A[s[i][j]] for j in R3)
        for j, k in itertools.product(R3, R3):
            conn = sum(G.C[l][s[j][i]] * A[s[k][l]] for l in R3)
            m = m + G.ig[s[j][k]] * (dA[j][s[k][i]] - conn
                                     - 1.5 / G.chi * A[s[k][i]] * G.dchi[j])
        out.append(m)
    return torch.stack(out)


def _padded(F, H, wrap):
    """F (24, n0, n1, n2) with H more points on every side: its edge values, or periodic ones."""
    for a in R3:
        n = F.shape[1 + a]
        i = torch.arange(-H, n + H, device=F.device)
        F = F.index_select(1 + a, i % n if wrap else i.clamp(0, n - 1))
    return F


def _by_slabs(fn, P, H, points=4_000_000):
    """fn(P, H) over slabs of x planes (bounds the temporaries of large grids)."""
    n = P.shape[-3] - 2 * H
    rows = max(1, points // ((P.shape[-2] - 2 * H) * (P.shape[-1] - 2 * H)))
    return torch.cat([fn(P[:, x:min(x + rows, n) + 2 * H], H) for x in range(0, n, rows)], dim=1)


def _enforce(F):
    """det(gt) = 1, tr(At) = 0, floors of chi and alpha."""
    F = F.clone()
    g = [F[GT + q] for q in range(6)]
    scale = _inverse(g)[1] ** (-1.0 / 3.0)
    g = [v * scale for v in g]
    ig, det = _inverse(g)
    tr = det * _contract(ig, [F[AT + q] for q in range(6)]) / 3.0
    for q in range(6):
        F[GT + q] = g[q]
        F[AT + q] = F[AT + q] - g[q] * tr
    F[CHI].clamp_(min=FLOOR)
    F[ALPHA].clamp_(min=FLOOR)
    return F


def _inner(F, ng):
    return F[(Ellipsis,) + (slice(ng, -ng),) * 3]


def _rk4(y, f, t, dt):
    """One classic step of y by the rate f(y, t) (no enforcement)."""
    k1 = f(y, t)
    k2 = f(y + 0.5 * dt * k1, t + 0.5 * dt)
    k3 = f(y + 0.5 * dt * k2, t + 0.5 * dt)
    k4 = f(y + dt * k3, t + dt)
    return y + (dt / 6.0) * (k1 + 2.0 * k2 + 2.0 * k3 + k4)


def _grid_rate(state, order, sigma, wrap):
    H = _ko_order(order) // 2 if sigma > 0.0 else order // 2
    h, dt = state["grid"].dx, state["dt"]

    def f(y, t):
        return _by_slabs(lambda P, H: _rates(P, H, h, dt, t, order, sigma), _padded(y, H, wrap),
                         H)
    return f


def _radiate(k, y, grid, order):
    """k with the rates of the ghost zones replaced by the outgoing-wave condition of y: face by
    face (x, y, z), one-sided along the normal, centred (edge values beyond) across."""
    ng, h = grid.ng, grid.dx
    R = order // 2
    X = [torch.as_tensor(c, device=y.device).view([-1 if b == a else 1 for b in R3])
         for a, c in enumerate((grid.x, grid.y, grid.z))]
    r = torch.sqrt(X[0] ** 2 + X[1] ** 2 + X[2] ** 2)
    r = torch.where(r == 0.0, torch.ones_like(r), r)
    P = _padded(y, R, False)
    S = _Stencils(P, R, h, order)
    k = k.clone()
    for f in range(NF):
        cen = [S.d1(f, a) for a in R3]
        for a in R3:
            for side in (0, 1):
                zone = [slice(None)] * 3
                zone[a] = slice(0, ng) if side == 0 else slice(y.shape[1 + a] - ng, None)
                zone = tuple(zone)
                d = list(cen)
                d[a] = (S._shift(f, a, 1) - S.at(f) if side == 0 else
                        S.at(f) - S._shift(f, a, -1)) / h
                k[f][zone] = (-(X[0] * d[0] + X[1] * d[1] + X[2] * d[2]) / r)[zone]
    return k


# MSRK rk4_2_2 coefficients
_A2 = (1309.0 / 15500.0, -31999.0 / 15500.0)
_A3 = (-241289.0 / 5880000.0, 22846301.0 / 16170000.0, -936169.0 / 2587200.0)
_B = (-191.0 / 882.0, 48241.0 / 59994.0, 193750.0 / 4351347.0, 100000.0 / 271791.0)


def _exact_evolution(state):
    case, grid, dt = state["case"], state["grid"], state["dt"]
    kind, order, ng = case["kind"], case["order"], state["grid"].ng
    U = state["U"].clone()
    if kind == "series":       # stage inputs synced, every padded point advanced, own ghosts kept
        rate = _grid_rate(state, order, 0.1, False)
        for s in range(case["steps"]):
            U = _enforce(_rk4(U, lambda y, t: rate(_padded(_inner(y, ng), ng, True), t), s * dt,
                              dt))
        C = _constraint_fields(_padded(U, order // 2, False), order // 2, grid.dx, order)
        return (U,) + _norms(C, ng)
    if kind == "radiative":
        rate = _grid_rate(state, order, 0.1, False)
        for s in range(case["steps"]):
            U = _enforce(_rk4(U, lambda y, t: _radiate(rate(y, t), y, grid, order), s * dt, dt))
        return U
    rate = _grid_rate(state, order, 0.1, True)
    y = _inner(U, ng)
    if kind == "rk4":
        for s in range(case["steps"]):
            y = _enforce(_rk4(y, rate, s * dt, dt))
        return _padded(y, ng, True)
    k0 = rate(y, 0.0)
    y = _enforce(_rk4(y, rate, 0.0, dt))
    for s in range(1, case["steps"]):
        t = s * dt
        k1 = rate(y, t)
        k2 = rate(y + dt * (_A2[0] * k0 + _A2[1] * k1), t + sum(_A2) * dt)
        k3 = rate(y + dt * (_A3[0] * k0 + _A3[1] * k1 + _A3[2] * k2), t + sum(_A3) * dt)
        y = _enforce(y + dt * (_B[0] * k0 + _B[1] * k1 + _B[2] * k2 + _B[3] * k3))
        k0 = k1
    return _padded(y, ng, True)


def _norms(C, ng):
    I = _inner(C, ng)
    return (float(torch.sqrt((I[0] ** 2).mean())),
            float(torch.sqrt((I[1] ** 2 + I[2] ** 2 + I[3] ** 2).mean())))


_MID = [3.0 / 256, -25.0 / 256, 150.0 / 256, 150.0 / 256, -25.0 / 256, 3.0 / 256]


def _refinement(fine, n):
    """The 1D 2:1 refinement as a matrix: rows the given fine indices, columns n coarse points
    (taps clamped to them)."""
    T = torch.zeros(len(fine), n, dtype=torch.float64)
    for row, p in enumerate(fine):
        if p % 2 == 0:
            T[row, p // 2] = 1.0
        else:
            for j, w in enumerate(_MID):
                T[row, min(max((p - 1) // 2 + j - 2, 0), n - 1)] += w
    return T.cuda()


def _refine3(F, T):
    """F (..., n0, n1, n2) refined along each axis by the matrices T."""
    F = torch.matmul(F, T[2].T.contiguous())
    F = torch.matmul(F.transpose(-1, -2).contiguous(), T[1].T.contiguous()) \
        .transpose(-1, -2).contiguous()
    lead, n = F.shape[:-3], F.shape[-3:]
    F = torch.matmul(T[0], F.reshape(-1, n[0], n[1] * n[2]))
    return F.reshape(*lead, T[0].shape[0], n[1], n[2])


def _hierarchy_step(levels, ng, fill, h, t, dt):
    """One shared-dt RK4 step of a list of padded level arrays (24, ..., S, S, S), ghosts of
    every stage input and of the result by fill(levels)."""
    H = 3

    def rate(Y, tt):
        m = ng - H
        return [_by_slabs(lambda P, H, q=q: _rates(P, H, h[q], dt, tt, 4, 0.1),
                          _inner(A, m) if m else A, H) if A.dim() == 4 else
                _rates(_inner(A, m) if m else A, H, h[q], dt, tt, 4, 0.1)
                for q, A in enumerate(Y)]

    def advanced(c, k):
        Y = [A.clone() for A in levels]
        for A, d in zip(Y, k):
            _inner(A, ng).add_(c * d)
        return Y

    k1 = rate(levels, t)
    k2 = rate(fill(advanced(0.5 * dt, k1)), t + 0.5 * dt)
    k3 = rate(fill(advanced(0.5 * dt, k2)), t + 0.5 * dt)
    k4 = rate(fill(advanced(dt, k3)), t + dt)
    new = advanced(dt / 6.0, [a + 2.0 * b + 2.0 * c + d
                              for a, b, c, d in zip(k1, k2, k3, k4)])
    for A in new:
        _inner(A, ng).copy_(_enforce(_inner(A, ng)))
    return fill(new)


def _exact_patches(state):
    H, U, ng = state["H"], state["U"], state["H"].ng
    levels = []
    for L, box in enumerate(H.boxes):
        A = torch.zeros([NF] + [e + 2 * ng for e in box.extent], dtype=torch.float64,
                        device=U.device)
        for b in range(len(H)):
            if H.level[b] == L:
                A[_patch_slices(H, b)] = H.view(U, b)
        levels.append(A)
    T = [None]
    for par, box in zip(H.boxes, H.boxes[1:]):
        T.append([_refinement([box.origin[a] - ng + i - 2 * (par.origin[a] - ng)
                               for i in range(box.extent[a] + 2 * ng)],
                              par.extent[a] + 2 * ng) for a in R3])

    def fill(Y):
        Y[0] = _padded(_inner(Y[0], ng), ng, True)
        for L in range(1, len(Y)):
            A = _refine3(Y[L - 1], T[L])
            _inner(A, ng).copy_(_inner(Y[L], ng))
            Y[L] = A
        return Y

    levels = _hierarchy_step(levels, ng, fill, [b.h for b in H.boxes], state["t"], state["dt"])
    out = U.clone()
    for b in range(len(H)):
        H.view(out, b).copy_(levels[H.level[b]][_patch_slices(H, b)])
    return out


def _exact_octree(state):
    H, U, ng, BS, W = (state["H"], state["U"], state["H"].ng, state["H"].BS, state["H"].W)
    tiles = [H.tree.on_level(L) for L in range(H.levels)]
    index = [{t: i for i, t in enumerate(ts)} for ts in tiles]
    levels = [torch.stack([H.view(U, t) for t in ts], dim=1) for ts in tiles]
    T = [_refinement([ng + c * BS + i for i in range(W)], W) for c in (0, 1)]

    def fill(Y):
        big = torch.zeros([NF] + [BS * r for r in H.nb_root], dtype=torch.float64,
                          device=U.device)
        for i, t in enumerate(tiles[0]):
            o = [BS * v for v in t[1:]]
            big[:, o[0]:o[0] + BS, o[1]:o[1] + BS, o[2]:o[2] + BS] = _inner(Y[0][:, i], ng)
        big = _padded(big, ng, True)
        for i, t in enumerate(tiles[0]):
            o = [BS * v for v in t[1:]]
            Y[0][:, i] = big[:, o[0]:o[0] + W, o[1]:o[1] + W, o[2]:o[2] + W]
        for L in range(1, len(Y)):
            own = [_inner(Y[L][:, i], ng).clone() for i in range(len(tiles[L]))]
            for i, t in enumerate(tiles[L]):
                par = (L - 1,) + tuple(v >> 1 for v in t[1:])
                A = _refine3(Y[L - 1][:, index[L - 1][par]], [T[v & 1] for v in t[1:]])
                for a, side in itertools.product(R3, (0, 1)):
                    n = list(t)
                    n[1 + a] += 1 if side else -1
                    j = index[L].get(tuple(n))
                    if j is not None:      # face slab over the interior extent
                        dst = [slice(ng, ng + BS)] * 3
                        src = [slice(None)] * 3
                        dst[a] = slice(ng + BS, W) if side else slice(0, ng)
                        src[a] = slice(0, ng) if side else slice(BS - ng, BS)
                        A[(slice(None),) + tuple(dst)] = own[j][(slice(None),) + tuple(src)]
                _inner(A, ng).copy_(own[i])
                Y[L][:, i] = A
        return Y

    levels = _hierarchy_step(levels, ng, fill, [H.spacing(L) for L in range(H.levels)],
                             state["t"], state["dt"])
    out = U.clone()
    for ts, A in zip(tiles, levels):
        for i, t in enumerate(ts):
            H.view(out, t).copy_(A[:, i])
    return out


def exact(case, seed):
    state = prepare(case, seed)
    kind = case["kind"]
    if kind == "patches":
        return _exact_patches(state)
    if kind == "octree":
        return _exact_octree(state)
    if kind == "rhs":
        return _grid_rate(state, case["order"], 0.0, False)(state["U"], state["t"])
    if kind == "constraints":
        H, order, h = case["order"] // 2, case["order"], state["grid"].dx
        C = _by_slabs(lambda P, H: _constraint_fields(P, H, h, order),
                      _padded(state["U"], H, False), H)
        return (C[0], C[1], C[2], C[3]) + _norms(C, state["grid"].ng)
    return _exact_evolution(state)
