"""Step bookkeeping (row sums, order sums, sequence statistics, normalization, Euler step),
transfers, roots and correlator launches at the edges of their work mapping, against the float64
oracle: sequence counts kept in registers (8) and read from memory (9, 17), reductions of 256 and
of 1024 threads, blocks of 2, 4 and 70 elements, more than 256 propagator rows, tables handed over
by a kernel and (beyond 64 KB) by a copy.  Tolerance 1e-10 relative, as for every float64 path; a
deviation's error is bounded by 1e-10 of the samples' scale."""
import ctypes as C

import numpy as np
import pytest

import oracle_lib as O
import qiw
from qiw import abi, model
from qiw.sobol import ScrambledSobolSeq

pytestmark = pytest.mark.gpu
RTOL = 1e-10
MODELS = {"level": lambda n_tau: model.bethe_single_level(n_tau, 10.0),
          "orbital": lambda n_tau: model.anderson_single_orbital(n_tau=n_tau),
          "blocks": lambda n_tau: model.kanamori(2, 2.0, 0.2, -1.0, 10.0, n_tau, 0.5)}


def rel(a, b):
    return np.linalg.norm((np.asarray(a) - np.asarray(b)).ravel()) / np.linalg.norm(np.asarray(b).ravel())


def std_close(s_gpu, s_cpu, mean_cpu):
    scale = np.abs(mean_cpu).max() + np.abs(s_cpu).max()
    return np.abs(np.asarray(s_gpu) - np.asarray(s_cpu)).max() <= RTOL * scale


@pytest.mark.parametrize("which,order,log2n,n_seqs,target", [
    ("level", 3, 5, 8, 0.0), ("level", 3, 5, 9, 0.0), ("orbital", 2, 6, 17, 1e-3), ("orbital", 3, 4, 8, 1e-3),
    ("blocks", 2, 2, 8, 1e-2), ("blocks", 1, 3, 9, 1e-3)])
def test_sequences(which, order, log2n, n_seqs, target):
    eg, ec = MODELS[which](8), MODELS[which](8)
    orders, N = range(0, order + 1), 2 ** log2n
    Po_g, Ps_g = qiw.inchworm(eg, eg.grid, orders, orders, N, rand_params=qiw.RandomizationParams(7, n_seqs, target))
    P_c, Po_c, Ps_c = O.inchworm(ec, orders, orders, N, rand=(n_seqs, 1, 7, target))
    assert rel(eg.P, P_c) < RTOL
    for o in orders:
        assert np.abs(Po_g[o] - Po_c[o]).max() < RTOL * np.abs(P_c).max()
        assert std_close(Ps_g[o], Ps_c[o], Po_c[o])


@pytest.mark.parametrize("which,n_tau,order,log2n", [("level", 4, 2, 16), ("orbital", 4, 1, 16), ("blocks", 4, 1, 9)])
def test_many_rows(which, n_tau, order, log2n):
    eg, ec = MODELS[which](n_tau), MODELS[which](n_tau)
    orders = range(0, order + 1)
    qiw.inchworm(eg, eg.grid, orders, orders, 2 ** log2n)
    P_c, Po_c, _ = O.inchworm(ec, orders, orders, 2 ** log2n)
    assert rel(eg.P, P_c) < RTOL


@pytest.mark.parametrize("which,n_tau", [("level", 300), ("blocks", 40), ("blocks", 130)])
def test_many_times(which, n_tau):
    eg, ec = MODELS[which](n_tau), MODELS[which](n_tau)
    qiw.inchworm(eg, eg.grid, range(0, 2), range(0, 2), 4)
    P_c, _, _ = O.inchworm(ec, range(0, 2), range(0, 2), 4)
    assert rel(eg.P, P_c) < RTOL
    eg, ec = MODELS[which](n_tau), MODELS[which](n_tau)
    S_g, _ = qiw.diff_inchworm(eg, eg.grid, range(1, 3), 4)
    P_c, S_c = O.diff_inchworm(ec, range(1, 3), 4)[:2]
    assert rel(eg.P, P_c) < RTOL


@pytest.mark.parametrize("n", range(1, 13))
def test_roots(n):
    """First simplex coordinate x^(1/n): half an ulp of the last rounding and up to one of the
    correction before it, against extended precision (0 and 1 ulp at x = 0)."""
    ctx, seq, N = qiw.context(), ScrambledSobolSeq(n), 4096
    ctx.check(ctx.lib.qiw_set_sobol(ctx.h, n, abi.ptr(np.ascontiguousarray(seq.m), C.c_uint32),
                                    abi.ptr(np.ascontiguousarray(seq.x0), C.c_uint32)))
    out = np.zeros((N, n))
    ctx.check(ctx.lib.qiw_simplex_points(ctx.h, 0, n, 0.0, 0.0, 1.0, N, out.ctypes.data_as(abi._f64p)))
    x = np.asarray(seq.points(N))[:, 0].astype(np.longdouble)
    y = np.where(x > 0, np.exp(np.log(np.where(x > 0, x, 1)) / n), 0)
    assert np.all(np.abs(out[:, 0] - y) <= 1.5 * np.spacing(np.maximum(out[:, 0], 2.0 ** -40)))


@pytest.mark.parametrize("order,log2n", [(0, 0), (1, 3), (2, 6), (3, 7), (4, 2)])
def test_pairs_together(order, log2n):
    """Correlators of several pairs in one launch (three pairs, and eight: every output of a
    wavefront in use) against the float64 oracle and against each pair alone."""
    for copies in (1, 3):
        e = model.anderson_single_orbital(n_tau=9, with_correlators=True)
        e = model.Expansion(e.ed, e.grid, e.pairs, (list(e.corr_operators) * copies)[:8])
        qiw.inchworm(e, e.grid, range(0, 2), range(0, 2), 16)
        orders, N = range(0, order + 1), 2 ** log2n
        g = qiw.correlator_2p(e, e.grid, orders, N)
        c = O.correlator_2p(e, orders, N)
        for i, x in enumerate(g):
            one = model.Expansion(e.ed, e.grid, e.pairs, [e.corr_operators[i]])
            one.P, one.P_n_known, one.P_der0 = e.P, e.P_n_known, e.P_der0
            alone = qiw.correlator_2p(one, one.grid, orders, N)[0]
            scale = np.abs(np.asarray(c[i])).max() + 1e-3
            assert np.abs(x - np.asarray(c[i])).max() < RTOL * scale
            assert np.abs(x - alone).max() < RTOL * scale
