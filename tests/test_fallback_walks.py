"""Models that the arc walks refuse run on the walks of the assignment tries: the kernel that is
launched for each, and the candidates of the work-mapping tuner, on a runtime that records
launches."""
import ctypes as C

import pytest

import qiw
from fallback_models import WALKS, F64, many_pairs, scaled_levels
from hip_stub import stub, stub_path  # noqa: F401
from qiw import abi
from test_gpu_arcs import fermions, parity, particles


@pytest.mark.parametrize("name", WALKS)
def test_kernel_of_a_refused_model(stub, name):  # noqa: F811
    kernel, make, order, prec = WALKS[name]
    orders = range(0, order + 1)
    stub.clear()
    qiw.inchworm_step(make(), 2, orders, 4, precision=prec, ctx=stub.ctx)
    names = [x.name for x in stub.launches("k_eval")]
    assert names and all(kernel in n for n in names)
    if name != "flat":  # (no group of these models fits; of the scaled levels only the bold ones do not)
        e = make()
        for call in (lambda: qiw.inchworm(e, e.grid, orders, orders, 4, precision=prec, ctx=stub.ctx),
                     lambda: qiw.correlator_2p(e, e.grid, orders, 4, precision=prec, ctx=stub.ctx)):
            stub.clear()
            call()
            names = [x.name for x in stub.launches("k_eval")]
            assert names and all(kernel in n for n in names)


# the candidates are those of the walk that the batch runs on, not of the one that was tried first
@pytest.mark.parametrize("make,order,prec,candidates", [
    (lambda: many_pairs(3, particles), 2, F64, 5),             # vector walk: chunk costs
    (lambda: fermions(3, particles), 2, F64, 7),               # arc walk: samples per workgroup
    (lambda: many_pairs(4, parity), 1, abi.QIW_PREC_FP32, 15),  # matrix-core walk: both
    (lambda: many_pairs(4, parity), 1, F64, 7),                # LDS block walk: samples per workgroup
    (scaled_levels, 4, F64, 7)])                               # flat walk: chunk words
def test_tuner_tries_the_walk_that_runs(stub, make, order, prec, candidates):  # noqa: F811
    e = make()
    qiw.inchworm_step(e, 2, range(0, order + 1), 4, precision=prec, ctx=stub.ctx)
    run, out = abi.RunStruct(list(range(0, order + 1)), [], 2 ** 6, 0, prec), abi.qiw_tuning()
    stub.ctx.check(stub.lib.qiw_autotune(stub.ctx.h, run.ref(), C.byref(out)))
    assert out.n_tried == candidates
