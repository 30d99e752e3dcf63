"""The walk a batch runs on (prefer_tries, qiw_host.cpp), by the kernel that is launched on a runtime
that records launches: the arc walk, but for few diagrams of small blocks on many samples (vector
walk) and of wide float64 blocks (LDS block walk).  The sizes are those whose times stand beside
the rule, at least a factor of two from its line."""
import pytest

import qiw
from hip_stub import stub, stub_path  # noqa: F401
from qiw import abi, model
from test_gpu_arcs import fermions, particles
from test_noalloc_limits import many_sectors

F64, F32 = abi.QIW_PREC_FP64, abi.QIW_PREC_FP32
ARC, VEC, BLOCK = "k_eval_arcs_t", "k_eval_vec_t", "k_eval_block"


def two_orbital(corr=False):
    e = model.kanamori(2, 2.0, 0.2, -1.0, 10.0, 12, 0.5)
    return model.Expansion(e.ed, e.grid, e.pairs, [(e.pairs[0].operator_i, e.pairs[0].operator_f)] if corr else [])


def blocks_of_three():
    return fermions(3, particles, 12)


@pytest.mark.parametrize("make,order,log2n,prec,kernel", [
    (two_orbital, 0, 0, F64, ARC), (two_orbital, 1, 0, F64, ARC), (two_orbital, 1, 12, F64, ARC), (two_orbital, 1, 18, F64, VEC),
    (two_orbital, 1, 18, F32, VEC), (two_orbital, 2, 18, F64, ARC), (two_orbital, 3, 12, F64, ARC),
    (blocks_of_three, 1, 18, F64, VEC), (blocks_of_three, 2, 9, F64, ARC), (blocks_of_three, 2, 18, F64, VEC),
    (blocks_of_three, 3, 12, F64, ARC), (lambda: many_sectors(12), 1, 9, F64, ARC), (lambda: many_sectors(12), 1, 13, F64, VEC),
    (lambda: fermions(5, particles, 12), 1, 15, F64, BLOCK), (lambda: fermions(5, particles, 12), 1, 15, F32, ARC),
    (lambda: fermions(5, particles, 12), 2, 12, F64, ARC)])
def test_walk_of_a_step(stub, make, order, log2n, prec, kernel):  # noqa: F811
    stub.clear()
    qiw.inchworm_step(make(), 3, range(0, order + 1), 2 ** log2n, precision=prec, ctx=stub.ctx)
    names = [x.name for x in stub.launches("k_eval")]
    assert names and all(kernel in n for n in names)


@pytest.mark.parametrize("order,log2n,kernel", [(1, 6, ARC), (1, 15, VEC), (2, 6, ARC)])
def test_walk_of_the_other_calls(stub, order, log2n, kernel):  # noqa: F811
    """Correlators count every tau row, the differential solve one."""
    e, orders = two_orbital(corr=True), range(0, order + 1)
    for call in (lambda: qiw.correlator_2p(e, e.grid, orders, 2 ** log2n, ctx=stub.ctx),
                 lambda: qiw.inchworm(e, e.grid, orders, orders, 2 ** (log2n + (3 if kernel == VEC else 0)), ctx=stub.ctx)):
        stub.clear()
        call()
        names = [x.name for x in stub.launches("k_eval")]
        assert names and all(kernel in n for n in names)
    stub.clear()
    qiw.diff_inchworm(e, e.grid, orders, 2 ** log2n, ctx=stub.ctx)
    assert all(ARC in x.name for x in stub.launches("k_eval"))  # (order 1 is one sample)


@pytest.mark.parametrize("log2n,kernel", [(13, ARC), (18, VEC)])
def test_walk_of_randomized_steps(stub, log2n, kernel):  # noqa: F811
    """Every sequence of a group counts: blocks of up to six at order 2 stay on the arc walk, of three
    do not."""
    for make, walk in ((two_orbital, ARC), (blocks_of_three, kernel)):
        stub.clear()
        qiw.inchworm_step(make(), 3, range(0, 3), 2 ** (log2n - 4), ctx=stub.ctx,
                          rand_params=qiw.RandomizationParams(5, 16 if make is two_orbital or kernel == VEC else 2, 0.0))
        names = [x.name for x in stub.launches("k_eval")]
        assert names and all(walk in n for n in names)
