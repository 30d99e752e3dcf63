"""The captured loop of bold steps (StepGraph, qiw_host.cpp) on a runtime that records launches:
a replay has to launch what the step-by-step loop launches for the same call (kernels, grids,
workgroups, LDS, arguments), whatever the context has solved before, and hold no device memory
that has been freed meanwhile."""
import pytest

import qiw
from hip_stub import stub, stub_path  # noqa: F401
from qiw import abi, model

WALKS = ("k_eval",)


def two_orbital(n_pairs, n_tau=8):
    e = model.kanamori(2, 2.0, 0.2, -1.0, 10.0, n_tau, 0.5)
    return model.Expansion(e.ed, e.grid, e.pairs[:n_pairs])


def single_orbital(n_pairs, n_tau=10):
    e = model.anderson_single_orbital(n_tau=n_tau)
    return model.Expansion(e.ed, e.grid, e.pairs[:n_pairs])


def solve_of(ctx, e, orders, N, prec):
    qiw.inchworm(e, e.grid, orders, orders, N, precision=prec, ctx=ctx)


def step_of(ctx, e, orders, N, prec):
    qiw.inchworm_step(e, 3, orders, N, precision=prec, ctx=ctx)


def solve(s, e, orders, N, prec):
    """The evaluator launches of a solve, and whether it was captured anew."""
    s.clear()
    solve_of(s.ctx, e, orders, N, prec)
    return s.launches(*WALKS), s.lib.stub_captures()


F64, F32 = abi.QIW_PREC_FP64, abi.QIW_PREC_FP32
# (make, orders, precision, calls): a call is (solve or step, pairs, samples); the last is a solve
SEQUENCES = {
    # programs for other workgroup shapes in the buffers of the first solve's plan
    "workgroup shape": (two_orbital, range(0, 4), F32, [("solve", 8, 2 ** 12), ("step", 8, 2 ** 5), ("solve", 4, 2 ** 12)]),
    # the operator table grows in between and its first buffer is freed
    "freed tables": (two_orbital, range(0, 2), F32, [("solve", 4, 2 ** 5), ("step", 8, 2 ** 5), ("solve", 4, 2 ** 5)]),
    "freed tables, float64": (two_orbital, range(0, 2), F64, [("solve", 4, 2 ** 5), ("step", 8, 2 ** 5), ("solve", 4, 2 ** 5)]),
    # a solve with fewer rows in LDS between the step and the solve with more
    "LDS": (single_orbital, range(0, 5), F64, [("step", 4, 2 ** 6), ("step", 4, 2 ** 5), ("solve", 2, 2 ** 6),
                                              ("step", 2, 2 ** 5), ("solve", 4, 2 ** 6)]),
}


@pytest.mark.parametrize("name", SEQUENCES)
def test_replay_launches_what_the_call_needs(stub, name):  # noqa: F811
    make, orders, prec, calls = SEQUENCES[name]
    for what, pairs, N in calls:
        if what == "step":
            step_of(stub.ctx, make(pairs), orders, N, prec)
        else:
            replayed, _ = solve(stub, make(pairs), orders, N, prec)
            assert all(x.freed == 0 for x in replayed)
    what, pairs, N = calls[-1]
    stub.ctx.check(stub.lib.qiw_set_graphs(stub.ctx.h, 0))
    eager, _ = solve(stub, make(pairs), orders, N, prec)
    stub.ctx.check(stub.lib.qiw_set_graphs(stub.ctx.h, 1))
    assert len(replayed) == len(eager) > 0
    for x, y in zip(replayed, eager):
        assert x[:4] == y[:4]
        assert x.args == y.args


def test_replay_of_an_unchanged_solve(stub):  # noqa: F811
    """The graph is kept while nothing changes: the second solve captures nothing."""
    for make, orders, prec in ((two_orbital, range(0, 3), F64), (single_orbital, range(0, 4), F64)):
        n = 8 if make is two_orbital else 4
        first, captured = solve(stub, make(n), orders, 2 ** 5, prec)
        again, recaptured = solve(stub, make(n), orders, 2 ** 5, prec)
        assert captured == 1 and recaptured == 0
        assert [x[:5] for x in first] == [x[:5] for x in again]


def test_first_solve_on_the_vector_walk_is_captured(stub):  # noqa: F811
    """Its tables are staged before the capture also where the bare step has another walk."""
    e = two_orbital(8)
    launched, captured = solve(stub, e, range(0, 2), 2 ** 17, F64)
    bold = [x for x in launched if "k_eval_vec_t" in x.name]
    assert captured == 1 and len(bold) >= e.grid.n_tau - 2
