"""Where QIW_PREC_FP32 has float32 chain products (include/qiw.h), by the instantiation of the
evaluator that is launched on a runtime that records launches."""
import pytest

import qiw
from hip_stub import stub, stub_path  # noqa: F401
from qiw import abi, model
from test_gpu_arcs import fermions, parity, particles


def many_tables(e):
    for i, p in enumerate(e.pairs):
        p.propagator = p.propagator * (1.0 + 0.1 * i)
    return e


@pytest.mark.parametrize("make,order,chains", [
    (lambda: fermions(3, particles), 4, "f"), (lambda: fermions(3, particles), 5, "d"),  # blocks up to 3
    (lambda: fermions(4, parity), 2, "f"), (lambda: many_tables(fermions(4, parity)), 2, "d"),  # up to 8; 4 tables
    (lambda: many_tables(fermions(3, particles)), 3, "f")])
def test_chains_of_a_float32_request(stub, make, order, chains):  # noqa: F811
    stub.clear()
    qiw.inchworm_step(make(), 2, range(0, order + 1), 4, precision=abi.QIW_PREC_FP32, ctx=stub.ctx)
    names = [x.name for x in stub.launches("k_eval")]
    assert names and all(f"k_eval_arcs_tI{chains}L" in n for n in names)
    stub.clear()
    qiw.inchworm_step(make(), 2, range(0, order + 1), 4, precision=abi.QIW_PREC_FP64, ctx=stub.ctx)
    assert all("k_eval_arcs_tIdL" in x.name for x in stub.launches("k_eval"))
