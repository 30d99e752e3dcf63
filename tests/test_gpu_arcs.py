"""The arc walk (k_eval_arcs_t) on sector blocks at the edges of its instantiations (largest
block 3, 8 | 16, 20 | 32), from one sample to several tasks per group, against the float64
oracle.  Tolerances as in the other block tests: 1e-10 relative in float64 (sums of the same
products in another order) and 2e-6 with float32 chain products."""
import numpy as np
import pytest

import oracle_lib as O
import qiw
from qiw import abi, model

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm((np.asarray(a) - np.asarray(b)).ravel()) / np.linalg.norm(np.asarray(b).ravel())


def fermions(n_modes, key, n_tau=6):
    """n_modes spinless levels with densities coupled and hopping between neighbours, every
    second one on a bath; sectors by key(basis state)."""
    fock = model.FockSpace(list(range(n_modes)))
    H = sum((0.1 * i - 0.3) * fock.n(i) for i in range(n_modes))
    for i in range(n_modes - 1):
        H = H + 0.4 * fock.n(i) @ fock.n(i + 1)
        t = fock.c_dag(i) @ fock.c(i + 1)
        H = H + 0.2 * (t + t.T)
    ed = model.EDCore(H, fock, key)
    grid = model.ImaginaryTimeGrid(5.0, n_tau)
    delta = 0.3 * model.bethe_gf(1.0, 5.0, grid)
    pairs = []
    for i in range(0, n_modes, 2):
        pairs.append(model.InteractionPair(fock.c_dag(i), fock.c(i), delta))
        pairs.append(model.InteractionPair(fock.c(i), fock.c_dag(i), model.ph_conj(delta)))
    return model.Expansion(ed, grid, pairs, [(-fock.c(0), fock.c_dag(0))])


def particles(b):
    return bin(b).count("1")


def parity(b):
    return bin(b).count("1") & 1


@pytest.mark.parametrize("precision", [abi.QIW_PREC_FP64, abi.QIW_PREC_FP32])
@pytest.mark.parametrize("n_modes,key,order,log2n", [(3, particles, 3, 0), (4, parity, 2, 4), (5, parity, 2, 1),
                                                     (6, particles, 1, 7), (6, parity, 1, 2), (3, particles, 4, 3),
                                                     (3, particles, 5, 1)])
def test_arc_walk(n_modes, key, order, log2n, precision):
    eg, ec = fermions(n_modes, key), fermions(n_modes, key)
    orders, N = range(0, order + 1), 2 ** log2n
    tol = 1e-10 if precision == abi.QIW_PREC_FP64 else 2e-6
    b_c, bo_c = O.inchworm_step_bare(ec, orders, N)
    if precision == abi.QIW_PREC_FP64:
        b_g, bo_g = qiw.inchworm_step_bare(eg, orders, N)
        assert rel(b_g, b_c) < tol and np.abs(bo_g - bo_c).max() < tol * np.abs(b_c).max()
    v_g, p_g = qiw.inchworm_step(eg, 2, orders, N, precision=precision)
    v_c, p_c = O.inchworm_step(ec, orders, N, 2)
    assert rel(v_g, v_c) < tol
    assert np.abs(p_g - p_c).max() < tol * np.abs(v_c).max()
    if order <= 3:
        g_g = qiw.correlator_2p(eg, eg.grid, orders, N, precision=precision)[0]
        g_c = O.correlator_2p(ec, orders, N)[0]
        assert rel(g_g, g_c) < tol


@pytest.mark.parametrize("log2n", [0, 6, 7])
@pytest.mark.parametrize("which,order", [("level", 6), ("orbital", 4), ("orbital", 1)])
def test_scalar_arc_walk(which, order, log2n):
    """The scalar arc walk (k_eval_sarcs_t) at its largest and smallest programs, one lane,
    one block and two blocks of samples, programs in few and in many segments."""
    make = (lambda: model.bethe_single_level(6)) if which == "level" else \
        (lambda: model.anderson_single_orbital(n_tau=6, with_correlators=True))
    eg, ec = make(), make()
    orders, N = range(0, order + 1), 2 ** log2n
    for words in (0, 64):
        qiw.set_tuning(chunk_words=words)
        try:
            b_g, _ = qiw.inchworm_step_bare(eg, range(0, min(order, 4) + 1), N)
            v_g, p_g = qiw.inchworm_step(eg, 2, orders, N)
            g_g = qiw.correlator_2p(eg, eg.grid, range(0, min(order, 3) + 1), N)
        finally:
            qiw.set_tuning()
        b_c, _ = O.inchworm_step_bare(ec, range(0, min(order, 4) + 1), N)
        v_c, p_c = O.inchworm_step(ec, orders, N, 2)
        assert rel(b_g, b_c) < 1e-10 and rel(v_g, v_c) < 1e-10
        assert np.abs(p_g - p_c).max() < 1e-10 * np.abs(v_c).max()
        for x, y in zip(g_g, O.correlator_2p(ec, range(0, min(order, 3) + 1), N)):
            assert rel(x, y) < 1e-10


@pytest.mark.parametrize("orders", [range(0, 1), range(0, 3)])
def test_model_without_pairs(orders):
    """A sector-block model that couples to no bath: the atomic propagator and correlator."""
    def make():
        e = fermions(3, particles)
        return model.Expansion(e.ed, e.grid, [], e.corr_operators)
    eg, ec = make(), make()
    assert rel(qiw.inchworm_step(eg, 2, orders, 4)[0], O.inchworm_step(ec, orders, 4, 2)[0]) < 1e-10
    assert rel(qiw.correlator_2p(eg, eg.grid, orders, 4)[0], O.correlator_2p(ec, orders, 4)[0]) < 1e-10


@pytest.mark.parametrize("n_modes", [3, 5])
def test_float32_sums_keep_small_terms(n_modes):
    """Float32 chain products, float64 sums (include/qiw.h): three pairs of the same operators whose
    hybridization functions are the constants 1, 2^-30 and -1 have the same chains, so order 1
    is 2^-30 times one of them to float32 accuracy.  Summed in float32 nothing of it is left.
    Blocks up to 3 and up to 10."""
    out = []
    for lib in (qiw, O):
        e = fermions(n_modes, particles)
        fock = model.FockSpace(list(range(n_modes)))
        one, small = (model.ScalarGF(np.full(e.grid.n_tau, -1j * v)) for v in (1.0, 2.0 ** -30))
        pairs = [model.InteractionPair(fock.c_dag(0), fock.c(0), one),
                 model.InteractionPair(fock.c_dag(0), fock.c(0), small),
                 model.InteractionPair(-fock.c_dag(0), fock.c(0), one)]
        e = model.Expansion(e.ed, e.grid, pairs)
        out.append(qiw.inchworm_step(e, 2, range(0, 2), 8, precision=abi.QIW_PREC_FP32) if lib is qiw
                   else O.inchworm_step(e, range(0, 2), 8, 2))
    (v_g, p_g), (v_c, p_c) = out
    assert rel(v_g, v_c) < 2e-6
    assert rel(p_g[1], p_c[1]) < 2e-6


def test_float32_requests_that_run_in_float64():
    """Orders beyond 4, and blocks wider than 6 with more than two hybridization functions, have
    float64 chains whatever is asked for."""
    def many_tables(e):
        for i, p in enumerate(e.pairs):
            p.propagator = p.propagator * (1.0 + 0.1 * i)
        return e
    for make, orders, N in ((lambda: fermions(3, particles), range(0, 6), 2),
                            (lambda: many_tables(fermions(5, particles)), range(0, 3), 4)):
        v_g, p_g = qiw.inchworm_step(make(), 2, orders, N, precision=abi.QIW_PREC_FP32)
        v_c, p_c = O.inchworm_step(make(), orders, N, 2)
        assert rel(v_g, v_c) < 1e-10
        assert np.abs(p_g - p_c).max() < 1e-10 * np.abs(v_c).max()
