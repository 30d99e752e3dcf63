"""Steps whose task rows come near the static scratch array of qiw_inchworm_step_noalloc, on a
runtime that records launches: the plan that inchworm_step leaves resident keeps its rows and the
other per-call buffers of the step within the array."""
import ctypes as C
import struct

import numpy as np
import pytest

import qiw
from hip_stub import stub, stub_path  # noqa: F401
from qiw import abi, model

F64, F32 = abi.QIW_PREC_FP64, abi.QIW_PREC_FP32


def three_orbital(n_tau):
    return model.kanamori(3, 3.0, 0.3, 0.0, 10.0, n_tau, 0.4)


def many_sectors(n_tau):
    """128 sectors of four states: 2048 elements in a row, blocks of the vector walk's sizes."""
    fock = model.FockSpace(list(range(9)))
    H = sum((0.1 * i - 0.3) * fock.n(i) for i in range(9))
    ed = model.EDCore(H, fock, lambda b: b >> 2)
    grid = model.ImaginaryTimeGrid(5.0, n_tau)
    delta = 0.3 * model.bethe_gf(1.0, 5.0, grid)
    pairs = [model.InteractionPair(fock.c_dag(8), fock.c(8), delta),
             model.InteractionPair(fock.c(8), fock.c_dag(8), model.ph_conj(delta))]
    return model.Expansion(ed, grid, pairs)


def noalloc(s, e, orders, N, precision):
    run = abi.RunStruct(list(orders), [], N, 0, precision)
    val = np.zeros(e.bt_size, np.complex128)
    per = np.zeros((len(orders), e.bt_size), np.complex128)
    return s.lib.qiw_inchworm_step_noalloc(s.ctx.h, run.ref(), 2, val.ctypes.data_as(abi._f64p),
                                           per.ctypes.data_as(abi._f64p))


def tables(launch):
    """Of an arc walk's launch: its tasks (group, first sample, first segment, segments), and the
    number of segments of each group's program."""
    groups, tasks, prog = struct.unpack_from("<3Q", launch.args)
    out, n_segments = [], {}
    for i in range(launch.grid[0]):
        g, sample, _, _, first, count = struct.unpack("<6i", C.string_at(tasks + 24 * i, 24))
        out.append((g, sample, first, count))
        prog_off = struct.unpack("<i", C.string_at(groups + 80 * g + 36, 4))[0]
        n_segments[g] = struct.unpack("<I", C.string_at(prog + 8 * prog_off, 4))[0]
    return out, n_segments


# a program in many segments (float64, cut by its first pairs), few samples; programs of seven
# segments; rows of many elements
CASES = [(three_orbital, 8, 3, 2 ** 6, F64), (three_orbital, 8, 3, 2 ** 7, F64), (three_orbital, 101, 2, 2 ** 8, F64),
         (three_orbital, 400, 3, 2 ** 7, F32), (many_sectors, 8, 1, 2 ** 12, F64), (many_sectors, 8, 1, 2 ** 12, F32),
         (many_sectors, 8, 1, 2 ** 9, F64), (many_sectors, 8, 1, 2 ** 9, F32)]


@pytest.mark.parametrize("make,n_tau,order,N,precision", CASES)
def test_rows_of_a_step_fit_the_scratch_array(stub, make, n_tau, order, N, precision):  # noqa: F811
    e, orders = make(n_tau), range(0, order + 1)
    stub.clear()
    qiw.inchworm_step(e, 2, orders, N, precision=precision, ctx=stub.ctx)
    resident = stub.launches("k_eval")
    stub.clear()
    rc = noalloc(stub, e, orders, N, precision)
    assert rc == abi.QIW_OK, stub.lib.qiw_last_error(stub.ctx.h).decode()
    launched = stub.launches("k_eval")
    assert [x[:4] for x in launched] == [x[:4] for x in resident]
    # every segment of a program is in one task of each sample block
    for x in launched:
        if "k_eval_arcs" not in x.name:
            continue
        tasks, n_segments = tables(x)
        blocks = {}
        for g, sample, first, count in tasks:
            blocks.setdefault((g, sample), []).append((first, count))
        for (g, _), parts in blocks.items():
            parts.sort()
            if parts != [(-1, 0)]:  # (the whole program)
                assert [p[0] for p in parts] == [0] + [p[0] + p[1] for p in parts[:-1]]
                assert sum(p[1] for p in parts) == n_segments[g] and min(p[1] for p in parts) > 0


def test_tuned_samples_per_workgroup_leave_the_rows_room(stub):  # noqa: F811
    """A setting that the vector walk did not look at: it must not refuse a step that was taken."""
    e, orders, N = many_sectors(8), range(0, 2), 2 ** 13
    qiw.inchworm_step(e, 2, orders, 2, ctx=stub.ctx)
    stub.ctx.check(stub.lib.qiw_set_tuning(stub.ctx.h, C.byref(abi.qiw_tuning(samples_per_task=1))))
    qiw.inchworm_step(e, 2, orders, N, ctx=stub.ctx)
    rc = noalloc(stub, e, orders, N, F64)
    assert rc == abi.QIW_OK, stub.lib.qiw_last_error(stub.ctx.h).decode()
