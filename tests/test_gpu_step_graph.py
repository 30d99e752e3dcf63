"""Solves whose loop of bold steps is replayed from a graph on a context that has run other
models meanwhile, against the step-by-step loop of the same call: the same kernels in the same
order, so the same bits."""
import numpy as np
import pytest

import qiw
from qiw import abi
from test_step_graph import SEQUENCES, solve_of, step_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", SEQUENCES)
def test_replay_equals_the_eager_loop(name):
    make, orders, prec, calls = SEQUENCES[name]
    ctx = abi.Context()
    try:
        for what, pairs, N in calls:
            print(f"{name}: {what}, {pairs} pairs, N={N}", flush=True)
            (solve_of if what == "solve" else step_of)(ctx, e := make(pairs), orders, N, prec)
        assert qiw.stats(ctx)["graph_replays"] > 0
        ctx.check(ctx.lib.qiw_set_graphs(ctx.h, 0))
        solve_of(ctx, f := make(pairs), orders, N, prec)
        assert np.array_equal(e.P, f.P)
    finally:
        ctx.close()
