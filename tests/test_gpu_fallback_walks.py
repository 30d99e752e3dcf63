"""The walks of the assignment tries on models that the arc walks refuse, against the float64
oracle: bare and bold steps, correlators, the differential solve, one sample to two blocks, and a
solve replayed from its graph.  Tolerances as for the arc walks on sector blocks: 1e-10 relative in
float64, 2e-6 with float32 chain products."""
import numpy as np
import pytest

import oracle_lib as O
import qiw
from fallback_models import F32, WALKS
from qiw import abi

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm((np.asarray(a) - np.asarray(b)).ravel()) / np.linalg.norm(np.asarray(b).ravel())


@pytest.mark.parametrize("log2n", [0, 3, 7])
@pytest.mark.parametrize("name", WALKS)
def test_refused_models(name, log2n):
    _, make, order, prec = WALKS[name]
    if name in ("matrix-core", "LDS block") and log2n > 3:
        log2n = 4  # (a wavefront per sample)
    orders, N, low = range(0, order + 1), 2 ** log2n, range(0, min(order, 2))
    tol = 2e-6 if prec == F32 else 1e-10
    eg, ec = make(), make()
    v_g, p_g = qiw.inchworm_step(eg, 2, orders, N, precision=prec)
    v_c, p_c = O.inchworm_step(ec, orders, N, 2)
    assert rel(v_g, v_c) < tol
    assert np.abs(p_g - p_c).max() < tol * np.abs(v_c).max()
    if prec != F32:
        assert rel(qiw.inchworm_step_bare(eg, orders, N)[0], O.inchworm_step_bare(ec, orders, N)[0]) < tol
    assert rel(qiw.correlator_2p(eg, eg.grid, low, N, precision=prec)[0], O.correlator_2p(ec, low, N)[0]) < tol
    qiw.diff_inchworm(eg, eg.grid, low, N, precision=prec)
    assert rel(eg.P, O.diff_inchworm(ec, low, N)[0]) < tol


@pytest.mark.parametrize("name", WALKS)
def test_replayed_solve(name):
    """The second solve stages nothing, so the vector and matrix-core walks run from a graph too; a
    step with fewer samples in between uses the same buffers."""
    _, make, order, prec = WALKS[name]
    orders = range(0, order if name != "flat" else order + 1)
    ctx = abi.Context()
    try:
        P = []
        for graphs in (1, 1, 0):
            ctx.check(ctx.lib.qiw_set_graphs(ctx.h, graphs))
            e = make()
            qiw.inchworm(e, e.grid, orders, orders, 8, precision=prec, ctx=ctx)
            P.append(e.P)
            assert (qiw.stats(ctx)["graph_replays"] > 0) == (graphs == 1 and name != "LDS block")
            qiw.inchworm_step(e, 2, orders, 4, precision=prec, ctx=ctx)
        assert np.array_equal(P[0], P[2]) and np.array_equal(P[1], P[2])
    finally:
        ctx.close()
