"""qiw_stats.n_kernel_launches against the evaluator launches a recording runtime sees: batches of
one and of several launches (one per workgroup shape), in steps, solves from a graph and one by one,
correlators and the differential solve."""
import pytest

import qiw
from hip_stub import stub, stub_path  # noqa: F401
from qiw import model

CALLS = {
    "step": lambda e, o, ctx: qiw.inchworm_step(e, 3, o, 16, ctx=ctx),
    "bare step": lambda e, o, ctx: qiw.inchworm_step_bare(e, o, 16, ctx=ctx),
    "solve": lambda e, o, ctx: qiw.inchworm(e, e.grid, o, o, 16, ctx=ctx),
    "correlator": lambda e, o, ctx: qiw.correlator_2p(e, e.grid, o, 16, ctx=ctx),
    "differential": lambda e, o, ctx: qiw.diff_inchworm(e, e.grid, o, 16, ctx=ctx),
}


@pytest.mark.parametrize("call", CALLS)
@pytest.mark.parametrize("which", ["orbital", "two orbitals"])
def test_launches_of_a_call(stub, which, call):  # noqa: F811
    if which == "orbital":
        e, orders = model.anderson_single_orbital(n_tau=9, with_correlators=True), range(0, 4)
    else:
        e, orders = model.kanamori(2, 2.0, 0.2, -1.0, 10.0, 9, 0.5), range(0, 4)
        e = model.Expansion(e.ed, e.grid, e.pairs, [(p.operator_i, p.operator_f) for p in e.pairs[:2]])
    for graphs in (1, 0):
        stub.ctx.check(stub.lib.qiw_set_graphs(stub.ctx.h, graphs))
        stub.clear()
        CALLS[call](e, orders, stub.ctx)
        assert qiw.stats(stub.ctx)["n_kernel_launches"] == len(stub.launches("k_eval")) > 0
