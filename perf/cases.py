"""Performance cases of the diagram-evaluation path: the calls a program makes when it solves
an impurity problem, through the package's public entry points (qiw.inchworm_step,
qiw.inchworm, qiw.correlator_2p, qiw.diff_inchworm).

Inputs follow self-consistent use: the local Hamiltonian of a case is fixed, while the bath
(hybridization strength) and the propagator table the call starts from change with the seed.
`exact` evaluates the same integrals in float64 with plain torch, by a recursion over the
configuration positions that keeps one value per set of open arcs.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qinchworm.jl_amd"))
import qiw  # noqa: E402
from qiw import abi, model  # noqa: E402


# ----------------------------------------------------------------------------------------
# The cases
# ----------------------------------------------------------------------------------------
# model: anderson (single orbital, 4 sectors of 1x1), bethe (one spinless level), kanamori2
#        (blocks 1 4 6 4 1), kanamori3 (blocks 1 6 15 20 15 6 1)
# call:  step, solve (inchworm!), corr (correlator_2p), diff (diff_inchworm!), rqmc (inchworm!
#        with several scrambled sequences)
# bath:  grid, spline or dlr (how the hybridization function is stored)
def _case(name, call, model_, n_tau, omax, log2n, fp32=False, bath="grid", n_w=0, n_seqs=1):
    c = {"call": call, "model": model_, "n_tau": n_tau, "omax": omax, "log2n": log2n, "fp32": fp32, "bath": bath,
         "n_w": n_w, "n_seqs": n_seqs}
    return dict(c, name=name) if name else c


def listed():
    return [
        # one bold step of a quick single-orbital run: latency of a call
        _case("anderson_step_small", "step", "anderson", 64, 2, 8, n_w=31),
        # a small solve with spline containers, as in the reference's own regression test
        _case("anderson_solve_spline", "solve", "anderson", 20, 3, 8, bath="spline"),
        # the single-orbital solve of the benchmark (float64, every bold step of the grid)
        _case("anderson_solve", "solve", "anderson", 200, 4, 14),
        # G, d and chi of the solved single-orbital model over the whole grid
        _case("anderson_corr", "corr", "anderson", 200, 3, 14),
        # the differential formulation on the same model
        _case("anderson_diff", "diff", "anderson", 200, 4, 13),
        # the randomized-qMC study: eight scrambled sequences per group
        _case("bethe_rqmc", "rqmc", "bethe", 200, 4, 12, n_seqs=8),
        # a high-order step of the single level on an odd grid
        _case("bethe_step_order5", "step", "bethe", 151, 5, 15, n_w=75),
        # a whole low-order solve of the two-orbital model in float64
        _case("kanamori2_solve", "solve", "kanamori2", 50, 2, 10),
        # a float64 step of the two-orbital model
        _case("kanamori2_step_fp64", "step", "kanamori2", 200, 3, 12, n_w=100),
        # the headline step (orders 0:4, float32 chain products) at a sample count that fits a pass
        _case("kanamori2_step_fp32", "step", "kanamori2", 200, 4, 11, fp32=True, n_w=100),
        # wide blocks in float64
        _case("kanamori3_step_fp64", "step", "kanamori3", 101, 2, 8, n_w=50),
        # wide blocks with float32 chain products
        _case("kanamori3_step_fp32", "step", "kanamori3", 400, 3, 9, fp32=True, n_w=200),
    ]


def draw(rng):
    """One more case of the same ranges; sizes over their logarithm, odd grids among them."""
    kind = rng.choice(["anderson", "anderson", "bethe", "kanamori2", "kanamori2", "kanamori3"])
    n_tau = int(round(math.exp(rng.uniform(math.log(20), math.log(200)))))
    if kind == "anderson":
        call = rng.choice(["step", "solve", "corr", "diff"])
        omax = rng.randint(1, 3 if call == "corr" else 4)
        log2n = rng.randint(5, 14 if call in ("step", "corr") else 12)
        bath = rng.choice(["grid", "grid", "spline"])
    elif kind == "bethe":
        call = rng.choice(["step", "rqmc", "corr"])
        omax = rng.randint(2, 5) if call == "step" else rng.randint(1, 4)
        log2n = rng.randint(5, 15 if call == "step" else 11)
        bath = "grid"
    elif kind == "kanamori2":
        call = rng.choice(["step", "step", "solve", "diff"])
        omax = rng.randint(1, 3) if call == "step" else rng.randint(1, 2)
        log2n = rng.randint(4, 11) if call == "step" else rng.randint(4, 8)
        bath = rng.choice(["grid", "grid", "dlr"])
    else:
        call, omax, bath = "step", rng.randint(1, 2), "grid"
        log2n = rng.randint(3, 7)
    fp32 = kind.startswith("kanamori") and rng.random() < 0.5
    n_w = rng.randint(1, n_tau - 2) if call == "step" else 0
    return _case(None, call, kind, n_tau, omax, log2n, fp32, bath, n_w, rng.choice([2, 3, 5]) if call == "rqmc" else 1)


# ----------------------------------------------------------------------------------------
# Inputs
# ----------------------------------------------------------------------------------------
BETA = {"anderson": 10.0, "bethe": 10.0, "kanamori2": 10.0, "kanamori3": 20.0}


@functools.lru_cache(maxsize=8)
def _local(kind, n_tau, spline, dlr):
    """The expansion with the family's own bath: the part of the inputs the seed leaves as it
    is (local Hamiltonian, operator blocks, grid)."""
    if kind == "anderson":
        return model.anderson_single_orbital(BETA[kind], n_tau, 0.1, 1.0, 0.5, 2.0, interpolate=spline, with_correlators=True)
    if kind == "bethe":
        return model.bethe_single_level(n_tau, BETA[kind])
    if kind == "kanamori2":
        return model.kanamori(2, 2.0, 0.2, -1.0, BETA[kind], n_tau, 0.5, interpolate=spline, dlr=dlr)
    return model.kanamori(3, 3.0, 0.3, 0.0, BETA[kind], n_tau, 0.4, interpolate=spline, dlr=dlr)


def _expansion(case, seed):
    """The expansion of a case: the local problem with a bath scaled by the seed and the
    propagator table a step or correlator starts from, i P_s(tau) = exp(-tau (E_s + lambda +
    M_s)) with small symmetric M_s (a dressed propagator with off-diagonal elements)."""
    base = _local(case["model"], case["n_tau"], case["bath"] == "spline", case["bath"] == "dlr")
    r = np.random.RandomState((seed * 7919 + 104729) % (1 << 31))
    e = model.Expansion.__new__(model.Expansion)
    e.__dict__.update(base.__dict__)
    scale = [r.uniform(0.8, 1.2) for _ in range(2)]  # occupied and empty parts of the bath apart
    e.pairs = [model.InteractionPair(p.operator_f, p.operator_i, p.propagator * scale[i % 2])
               for i, p in enumerate(base.pairs)]
    lam = base._lambda()
    P = np.zeros((case["n_tau"], base.bt_size), np.complex128)
    for s, E in enumerate(base.ed.energies):
        d = len(E)
        a = r.uniform(-0.05, 0.05, (d, d))
        w, U = np.linalg.eigh(np.diag(E + lam) + 0.5 * (a + a.T))
        blocks = np.einsum("ik,tk,jk->tij", U, np.exp(-base.grid.tau[:, None] * w[None, :]), U)
        o = base.bt_offsets[s]
        P[:, o:o + d * d] = -1j * blocks.transpose(0, 2, 1).reshape(case["n_tau"], d * d)
    if case["call"] in ("step", "corr"):
        e.P, e.P_n_known = P, case["n_tau"]
    else:  # the solvers start from the atomic propagator
        e.P = base.P.copy()
    e.P_der0 = base.P_der0.copy()
    return e


def prepare(case, seed):
    return {"case": case, "exp": _expansion(case, seed), "seed": seed, "orders": range(0, case["omax"] + 1),
            "N": 2 ** case["log2n"], "prec": abi.QIW_PREC_FP32 if case["fp32"] else abi.QIW_PREC_FP64}


def _typed(case, out):
    """Results of float32 chain products are kept in the type they are computed in."""
    if not case["fp32"]:
        return out
    return {k: (v.astype(np.complex64) if isinstance(v, np.ndarray) else {o: x.astype(np.complex64) for o, x in v.items()})
            for k, v in out.items()}


def run(state):
    c, e, orders, N, prec = state["case"], state["exp"], state["orders"], state["N"], state["prec"]
    if c["call"] == "step":
        val, per = qiw.inchworm_step(e, c["n_w"], orders, N, precision=prec)
        return _typed(c, {"value": val, "orders": per})
    if c["call"] == "solve":
        Po, _ = qiw.inchworm(e, e.grid, orders, orders, N, precision=prec)
        return _typed(c, {"P": e.P, "orders": Po})
    if c["call"] == "rqmc":
        rp = qiw.RandomizationParams(state["seed"], c["n_seqs"], 0.0)
        Po, Ps = qiw.inchworm(e, e.grid, orders, orders, N, precision=prec, rand_params=rp)
        return _typed(c, {"P": e.P, "orders": Po, "std": Ps})
    if c["call"] == "diff":
        So, _ = qiw.diff_inchworm(e, e.grid, orders, N, precision=prec)
        return _typed(c, {"P": e.P, "sigma": So})
    g = qiw.correlator_2p(e, e.grid, orders, N, precision=prec)
    return _typed(c, {"corr%d" % i: v for i, v in enumerate(g)})


# ----------------------------------------------------------------------------------------
# The recursion over open arcs: reference values and the work a pass cannot do without
# ----------------------------------------------------------------------------------------
def _maps(e):
    """Per pair the sector maps of its two operators, and the hybridization table."""
    ns = len(e.ed.dims)
    opi = [[ops[0][s][0] if s in ops[0] else -1 for s in range(ns)] for ops in e.pair_operator_mat]
    opf = [[ops[1][s][0] if s in ops[1] else -1 for s in range(ns)] for ops in e.pair_operator_mat]
    return ns, opi, opf


def _stages(e, kind, order, n_after, s0, corr=None):
    """Stages of one group and initial sector: per configuration position 2 .. n - 1 the pairs
    (source state, destination state, operator, sign, opened at) that join the states before
    and after it.  A state is (sector, open arcs as (point, pair), components of the arcs not
    yet joined to one across tau_w, number of joined arcs)."""
    ns, opi, opf = _maps(e)
    n_pts = 2 * order
    nb = {"bare": 0, "sigma": n_pts - 1}.get(kind, n_pts - n_after)  # points before the cut
    pos_w = {"bare": -1, "sigma": n_pts}.get(kind, n_pts - n_after)   # points before tau_w
    s = s0
    if kind == "corr":
        A, B = e.corr_operators_mat[corr]
        if s0 not in B:
            return None
        s = B[s0][0]
    level, steps = {(s, (), (), 0)}, []

    def cross():  # the node at tau_w
        out = set()
        joins = []
        for st in level:
            s2 = st[0]
            if kind == "corr":
                if st[0] not in A:
                    continue
                s2 = A[st[0]][0]
            d = (s2,) + st[1:]
            joins.append((st, d, "A" if kind == "corr" else None, 1, None))
            out.add(d)
        steps.append(joins)
        return out

    for j in range(n_pts):
        if j == pos_w:
            level = cross()
        rem, joins, out = n_pts - j, [], set()
        for st in level:
            s1, arcs, comp, good = st
            if j == nb:  # every arc open across the cut is joined
                comp, good = (), len(arcs)
            if len(arcs) + 1 <= rem - 1:
                for p in range(len(opi)):
                    if opi[p][s1] >= 0:
                        full = good if kind != "bare" else len(arcs) + 1
                        nc = () if kind == "bare" else comp + ((comp[-1] + 1) if comp else 0,)
                        d = (opi[p][s1], arcs + ((j, p),), nc, full)
                        joins.append((st, d, ("i", p), 1, None))
                        out.add(d)
            for i, (h, p) in enumerate(arcs):
                s2 = opf[p][s1]
                if s2 < 0:
                    continue
                rest = arcs[:i] + arcs[i + 1:]
                if i < good:  # later arcs cross it: all joined (bare: every arc counts as joined)
                    nc, ng = (), len(rest)
                else:
                    c = list(comp)
                    own = c[i - good]
                    c[i - good:] = [own] * (len(c) - (i - good))
                    del c[i - good]
                    if own not in c:
                        continue
                    names = {}
                    nc, ng = tuple(names.setdefault(x, len(names)) for x in c), good
                d = (s2, rest, nc, ng)
                joins.append((st, d, ("f", p), -1 if (len(arcs) - 1 - i) % 2 else 1, h))
                out.add(d)
        steps.append(joins)
        level = out
    if pos_w == n_pts:
        level = cross()
    # keep what reaches the closing state
    alive = {d for d in level if not d[1] and d[0] == s0}
    for k in range(len(steps) - 1, -1, -1):
        steps[k] = [x for x in steps[k] if x[1] in alive]
        alive = {x[0] for x in steps[k]}
    return steps if alive else None


def _groups(kind, orders, N):
    for k in orders:
        if kind == "sigma":
            if k > 0:
                yield k, 1
        elif kind == "bare" or k == 0:
            yield k, 2 * k if kind == "bare" else 0
        else:
            for na in range(1, 2 * k):
                yield k, na


@functools.lru_cache(maxsize=None)
def _group_flops(model_, kind, k, na, corr):
    e = _local(model_, 20, False, False)
    dims, fl = e.ed.dims, 0.0
    for s0 in range(len(dims)):
        steps = _stages(e, kind, k, na, s0, corr)
        for joins in steps or []:
            for s in {x[0]: None for x in joins}:
                fl += 2.0 * dims[s[0]] ** 2 * dims[s0]          # propagator
            for d, s, op in {(x[1], x[0][0], x[2]) for x in joins if x[2]}:
                fl += 2.0 * dims[d[0]] * dims[s] * dims[s0]     # operator
            fl += sum(2.0 * dims[x[0][0]] * dims[s0] for x in joins if x[4] is not None)  # arc
        if steps:
            fl += 2.0 * dims[s0] ** 3
    return fl


def work(case):
    e = _local(case["model"], case["n_tau"], case["bath"] == "spline", case["bath"] == "dlr")
    N, nt, bt = 2 ** case["log2n"], case["n_tau"], e.bt_size
    orders = range(case["omax"] + 1)

    def launch(kind, corr=None):
        return sum(_group_flops(case["model"], kind, k, na, corr) *
                   (1 if k == 0 or (kind == "sigma" and k == 1) else N) for k, na in _groups(kind, orders, N))
    tables = 16.0 * nt * len(e.pairs)
    out = 16.0 * bt * (case["omax"] + 2)
    if case["call"] == "step":
        return {"flops": launch("bold"), "bytes": tables + 16.0 * nt * bt + out}
    if case["call"] in ("solve", "rqmc"):
        n = case["n_seqs"]
        return {"flops": n * (launch("bare") + (nt - 2) * launch("bold")), "bytes": tables + nt * out}
    if case["call"] == "diff":
        return {"flops": (nt - 1) * launch("sigma") + sum(2.0 * d ** 3 for d in e.ed.dims) * nt * nt / 2,
                "bytes": tables + nt * out}
    nc = len(e.corr_operators)
    return {"flops": (nt - 1) * sum(launch("corr", i) for i in range(nc)),
            "bytes": tables + 16.0 * nt * bt + 16.0 * nt * nc}


class _Exact:
    """float64 evaluation of the same sums, batched over samples and states."""

    def __init__(self, case, e):
        self.dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
        self.e, self.n_tau, self.beta = e, case["n_tau"], e.grid.beta
        self.h = self.beta / (self.n_tau - 1)
        self.dims, self.off = e.ed.dims, [int(o) for o in e.bt_offsets]
        self.N, self.plans = 2 ** case["log2n"], {}
        self.E = [np.asarray(E) + e._lambda() for E in e.ed.energies]
        self.bath = {}
        for i, p in enumerate(e.pairs):
            g = p.propagator
            if g.kind == abi.QIW_GF_DLR:
                key = ("dlr", tuple(g.omega), tuple(g.coef))
            else:
                key = (g.kind, tuple(-np.asarray(g.values).imag))
            self.bath.setdefault(key, []).append(i)
        self.table_of = {p: t for t, ps in enumerate(self.bath.values()) for p in ps}
        self.tabs = [self._table(key) for key in self.bath]
        self.scalar = max(self.dims) == 1

    def t(self, x, dtype=torch.float64):
        return torch.as_tensor(np.ascontiguousarray(x), dtype=dtype, device=self.dev)

    def _table(self, key):
        if key[0] == "dlr":
            return ("dlr", self.t(np.array(key[1])), self.t(-np.array(key[2]).imag))
        y = np.array(key[1])
        if key[0] == abi.QIW_GF_GRID_LINEAR:
            return ("grid", self.t(y))
        n = len(y)  # natural cubic spline: second derivatives M
        A = np.diag(np.full(n - 2, 4.0)) + np.diag(np.ones(n - 3), 1) + np.diag(np.ones(n - 3), -1)
        M = np.zeros(n)
        M[1:-1] = np.linalg.solve(A, 6.0 * (y[2:] - 2.0 * y[1:-1] + y[:-2]))
        return ("spline", self.t(y), self.t(M))

    def cell(self, t1, t2):
        t1 = torch.maximum(t1, t2)
        x1, x2 = t1 / self.h, t2 / self.h
        i1, i2 = x1.floor().clamp(0, self.n_tau - 2), x2.floor().clamp(0, self.n_tau - 2)
        a, b = x1 - i1, x2 - i2
        return (i1 - i2).long(), a * (1 - b), (1 - a) * b

    def lookup(self, tab, cell):
        d, wp, wm = cell
        g0, gp = tab[d], tab[d + 1]
        gm = torch.where((d > 0).reshape(d.shape + (1,) * (tab.dim() - 1)), g0 - tab[(d - 1).clamp(min=0)], gp - g0)
        s = d.shape + (1,) * (tab.dim() - 1)
        return g0 + wp.reshape(s) * (gp - g0) - wm.reshape(s) * gm

    def delta(self, k, t1, t2):
        tab = self.tabs[k]
        if tab[0] == "grid":
            return self.lookup(tab[1], self.cell(t1, t2))
        z = (t1 - t2).clamp(min=0.0)
        if tab[0] == "dlr":
            w, out = tab[1], torch.zeros_like(z)
            for wk, ck in zip(w.tolist(), tab[2].tolist()):
                f = torch.exp(-wk * z) / (1 + math.exp(-wk * self.beta)) if wk >= 0 else \
                    torch.exp(wk * (self.beta - z)) / (1 + math.exp(wk * self.beta))
                out += ck * f
            return out
        x = z / self.h
        j = x.floor().clamp(0, self.n_tau - 2).long()
        u, y, M = x - j, tab[1], tab[2]
        return y[j] * (1 - u) + y[j + 1] * u + ((1 - u) ** 3 - (1 - u)) * M[j] / 6 + (u ** 3 - u) * M[j + 1] / 6

    @functools.lru_cache(maxsize=None)
    def points(self, d):
        if d == 0:
            return torch.zeros((self.N, 0), dtype=torch.float64, device=self.dev)
        eng = torch.quasirandom.SobolEngine(d, scramble=False)
        return eng.draw(self.N, dtype=torch.float64).to(self.dev)

    def times(self, kind, k, na, tw, tf):
        """Times of the configuration positions 1 .. n, each [N] (or [1] for exact groups), and
        the prefactor of the sample sum."""
        one = torch.ones(1, dtype=torch.float64, device=self.dev)
        if k == 0:
            return ([0 * one, tf * one] if kind == "bare" else [0 * one, tw * one, tf * one]), 1.0

        def root(x, lo, hi):  # descending times of the simplex on [lo, hi]
            out, prev = [], None
            for i in range(x.shape[1]):
                f = x[:, i] ** (1.0 / (x.shape[1] - i))
                prev = f if prev is None else prev * f
                out.append(lo + prev * (hi - lo))
            return out
        vol = lambda d, e: float(np.prod([e / i for i in range(1, d + 1)]))  # noqa: E731
        if kind == "sigma":
            x = self.points(2 * k - 2) if k > 1 else torch.zeros((1, 0), dtype=torch.float64, device=self.dev)
            o = torch.ones(x.shape[0], dtype=torch.float64, device=self.dev)
            before = [tw * o] + root(x, 0.0, tw) + [0 * o]
            return [0 * o] + before[::-1] + [tw * o, tf * o], vol(2 * k - 2, tw) / x.shape[0]
        x = self.points(2 * k)
        o = torch.ones(self.N, dtype=torch.float64, device=self.dev)
        after = root(x[:, :na], tw, tf)
        if kind == "bare":
            return [0 * o] + after[::-1] + [tf * o], vol(2 * k, tf) / self.N
        before = root(x[:, na:], 0.0, tw)
        return [0 * o] + before[::-1] + [tw * o] + after[::-1] + [tf * o], vol(2 * k - na, tw) * vol(na, tf - tw) / self.N

    def prop(self, kind, P, t1, t2):
        """i P per sector between two positions, [N, m, m] each ([ns, N] for 1x1 sectors)."""
        if kind == "bare":
            dt = (t1 - t2).clamp(min=0.0)
            if self.scalar:
                return torch.stack([torch.exp(-dt * float(E[0])) for E in self.E])
            return [torch.diag_embed(torch.exp(-dt[:, None] * self.t(E)[None, :])) for E in self.E]
        v = self.lookup(P, self.cell(t1, t2))
        if self.scalar:
            return v.T
        return [v[:, o:o + m * m].reshape(-1, m, m).transpose(1, 2) for o, m in zip(self.off, self.dims)]

    def block(self, op, s, corr):
        if op == "A":
            return self.e.corr_operators_mat[corr][0][s][1]
        ops = self.e.pair_operator_mat[op[1]][0 if op[0] == "i" else 1]
        return ops[s][1]

    def plan(self, kind, k, na, corr):
        """Index arrays of a group: for 1x1 sectors all initial sectors together, else one plan
        per initial sector with the operator products grouped by (operator, sector)."""
        key = (kind, k, na, corr)
        if key in self.plans:
            return self.plans[key]
        out = []
        pos_w = {"bare": -1, "sigma": 2 * k}.get(kind, 2 * k - na)
        pos_of = lambda j: 1 + j + (1 if 0 <= pos_w <= j else 0)  # noqa: E731  point -> position index (0-based)
        starts = []
        for s0 in range(len(self.dims)):
            st = _stages(self.e, kind, k, na, s0, corr)
            if st is None:
                if k > 0 or kind == "corr":
                    continue
                st = [] if kind == "bare" else [[((s0, (), (), 0), (s0, (), (), 0), None, 1, None)]]
            starts.append((s0, st))
        n_steps = 2 * k + (0 if kind == "bare" else 1)
        if self.scalar:
            first, idx, rows = [], {}, []
            for s0, st in starts:
                b = float(np.real(self.e.corr_operators_mat[corr][1][s0][1][0, 0])) if kind == "corr" else 1.0
                s = self.e.corr_operators_mat[corr][1][s0][0] if kind == "corr" else s0
                idx[(s0, (s, (), (), 0))] = len(first)
                first.append((s, b))
            for n in range(n_steps):
                src, dst, cf, arc, new = [], [], [], [], {}
                for s0, st in starts:
                    for x in st[n]:
                        v = 1.0 if x[2] is None else float(np.real(self.block(x[2], x[0][0], corr)[0, 0]))
                        src.append(idx[(s0, x[0])])
                        dst.append(new.setdefault((s0, x[1]), len(new)))
                        cf.append(v * x[3])
                        arc.append((pos_of(x[4]), self.table_of[x[2][1]]) if x[4] is not None else None)
                keys = sorted(set(a for a in arc if a), key=str)
                col = [keys.index(a) + 1 if a else 0 for a in arc]
                rows.append((self.t(src, torch.long), self.t(dst, torch.long), self.t(cf), keys, self.t(col, torch.long),
                             self.t([q[1][0] for q in new], torch.long), len(new)))
                idx = new
            last = self.t([s0 for s0, _ in idx], torch.long)
            out = (self.t([f[0] for f in first], torch.long), self.t([f[1] for f in first]), rows, last)
        else:
            for s0, st in starts:
                s = self.e.corr_operators_mat[corr][1][s0][0] if kind == "corr" else s0
                root = np.real(self.e.corr_operators_mat[corr][1][s0][1]) if kind == "corr" else np.eye(self.dims[s0])
                idx, rows = {(s, (), (), 0): (s, 0)}, []
                for n in range(n_steps):
                    new, count, by = {}, {}, {}
                    for x in st[n]:
                        if x[1] not in new:
                            d = x[1][0]
                            new[x[1]] = (d, count.get(d, 0))
                            count[d] = count.get(d, 0) + 1
                        by.setdefault((x[2], x[0][0], x[1][0], x[4]), []).append((idx[x[0]][1], new[x[1]][1], x[3]))
                    ops = []
                    for (op, ss, sd, h), v in by.items():
                        v = np.array(v)
                        O = None if op is None else self.t(np.real(self.block(op, ss, corr)))
                        ops.append((O, ss, sd, None if h is None else (pos_of(h), self.table_of[op[1]]),
                                    self.t(v[:, 0], torch.long), self.t(v[:, 1], torch.long), self.t(v[:, 2])))
                    rows.append((ops, count))
                    idx = new
                out.append((s0, s, self.t(root), rows))
        self.plans[key] = out
        return out

    def group(self, kind, k, na, tw, tf, P, corr=None):
        """Prefactor-weighted sum over samples of one group, in the block-table layout."""
        sign = -1.0 if kind == "corr" and na % 2 else 1.0
        tt, fac = self.times(kind, k, na, tw, tf)
        res = torch.zeros(int(self.e.bt_size), dtype=torch.float64, device=self.dev)
        plan, n, arcs = self.plan(kind, k, na, corr), len(tt), {}

        def arc(L, key, lo, hi):
            q = (L,) + key
            if q not in arcs:
                arcs[q] = self.delta(key[1], tt[L], tt[key[0]])
            return arcs[q][lo:hi]
        M = tt[0].shape[0]
        if self.scalar:
            first, val, rows, last = plan
            if not len(first):
                return res
            X = val[:, None] * self.prop(kind, P, tt[1], tt[0])[first] if n > 1 else val[:, None]
            for L, (src, dst, cf, keys, col, sec, m) in enumerate(rows, start=1):
                D = torch.stack([torch.ones(M, dtype=torch.float64, device=self.dev)] + [arc(L, q, 0, M) for q in keys])
                X = torch.zeros((m, M), dtype=torch.float64, device=self.dev).index_add_(0, dst, X[src] * (cf[:, None] * D[col]))
                X = X * self.prop(kind, P, tt[L + 1], tt[L])[sec]
            res.index_add_(0, last, X.sum(1))
            return sign * fac * res
        step = max(1, min(M, 1 << (8 if max(self.dims) <= 6 else 5)))
        for lo in range(0, M, step):
            hi = min(M, lo + step)
            props = [self.prop(kind, P, tt[L][lo:hi], tt[L - 1][lo:hi]) for L in range(1, n)]
            for s0, s, root, rows in plan:
                c = self.dims[s0]
                X = {s: (props[0][s] @ root)[None]}
                for L, (ops, count) in enumerate(rows, start=1):
                    Y = {d: torch.zeros((q, hi - lo, self.dims[d], c), dtype=torch.float64, device=self.dev)
                         for d, q in count.items()}
                    for O, ss, sd, h, src, dst, sg in ops:
                        w = sg[:, None] if h is None else sg[:, None] * arc(L, h, lo, hi)[None, :]
                        v = X[ss][src] * w[:, :, None, None]
                        Y[sd].index_add_(0, dst, v if O is None else torch.matmul(O, v))
                    X = {d: torch.matmul(props[L][d][None], y) for d, y in Y.items()}
                o = self.off[s0]
                res[o:o + c * c] += X[s0][0].sum(0).T.reshape(-1)
        return sign * fac * res

    def orders_sum(self, kind, orders, tw, tf, P, corr=None):
        per = {k: torch.zeros(int(self.e.bt_size), dtype=torch.float64, device=self.dev) for k in orders}
        for k, na in _groups(kind, orders, self.N):
            if not (kind == "sigma" and k > 1 and tw == 0.0):
                per[k] += self.group(kind, k, na, tw, tf, P, corr)
        return per


def _as_P(x):
    return -1j * x.cpu().numpy()


def exact(case, seed):
    if case["call"] == "rqmc":
        return None
    cost = work(case)["flops"]
    if case["call"] in ("solve", "diff") and (case["omax"] > 3 and case["n_tau"] > 100 or cost > 3e12):
        return None
    e = _expansion(case, seed)
    x = _Exact(case, e)
    orders, n_tau, h = list(range(case["omax"] + 1)), case["n_tau"], x.h
    diag = [o + i * (m + 1) for o, m in zip(x.off, x.dims) for i in range(m)]
    P = x.t(-np.asarray(e.P).imag)
    if case["call"] == "step":
        per = x.orders_sum("bold", orders, case["n_w"] * h, (case["n_w"] + 1) * h, P)
        return {"value": _as_P(sum(per.values())), "orders": np.stack([_as_P(per[k]) for k in orders])}
    if case["call"] == "corr":
        Z, out = float(P[-1, diag].sum()), {}
        for i in range(len(e.corr_operators)):
            v = np.zeros(n_tau)
            for j in range(n_tau):
                per = x.orders_sum("corr", orders if j else [0], j * h, x.beta, P, i)
                v[j] = float(sum(p[diag].sum() for p in per.values()))
            out["corr%d" % i] = -1j * v / Z
        return out
    tab = {k: torch.zeros((n_tau, int(e.bt_size)), dtype=torch.float64, device=x.dev) for k in orders}
    if case["call"] == "diff":
        shift = 1 if e.interpolate_ppgf else 0
        S = torch.zeros((n_tau + 1, int(e.bt_size)), dtype=torch.float64, device=x.dev)
        blocks = lambda T, o, m: T[:, o:o + m * m].reshape(-1, m, m).transpose(1, 2)  # noqa: E731
        for a in range(n_tau - 1):
            per = x.orders_sum("sigma", orders, a * h, a * h, P)
            for k in orders:
                tab[k][a + 1] = per[k]
            S[a + shift] = sum(per.values())
            for E, o, m in zip(x.E, x.off, x.dims):
                w = torch.full((a + 1,), h, dtype=torch.float64, device=x.dev)
                w[0] = w[a] = 0.5 * h
                c = torch.einsum("j,jab,jbc->ac", w, blocks(S[:a + 1].flip(0), o, m), blocks(P[:a + 1], o, m)) if a else 0.0
                p = blocks(P[a:a + 1], o, m)[0]
                P[a + 1, o:o + m * m] = (p + h * (c - x.t(E)[:, None] * p)).T.reshape(-1)
        return {"P": _as_P(P), "sigma": {k: 1j * tab[k].cpu().numpy() for k in orders}}
    for jf in range(1, n_tau):
        per = x.orders_sum("bare" if jf == 1 else "bold", orders, 0.0 if jf == 1 else (jf - 1) * h, jf * h, P)
        for k in orders:
            tab[k][jf] = per[k]
        P[jf] = sum(per.values())
        if jf > 1:
            lam = torch.log(P[jf, diag].max()) / (jf * h)
            known = jf + 1 if e.interpolate_ppgf else n_tau
            P[:known] *= torch.exp(-x.t(e.grid.tau[:known]) * lam)[:, None]
    return {"P": _as_P(P), "orders": {k: _as_P(tab[k]) for k in orders}}
