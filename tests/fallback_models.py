"""Small models that the arc walks refuse, one for each walk of the assignment tries: more
interaction pairs than a sector-block program can name (127), and a scalar model whose arc values
take more rows than the scalar walk has."""
from qiw import abi, model
from test_gpu_arcs import fermions, parity, particles


def many_pairs(n_modes, key, n_pairs=128):
    e = fermions(n_modes, key, n_tau=8)
    return model.Expansion(e.ed, e.grid, [e.pairs[i % len(e.pairs)] for i in range(n_pairs)], e.corr_operators)


def scaled_levels():
    """Three levels with four hybridization functions and operator elements other than one: 28 arcs
    of order 4 with a row per function and another per function and element."""
    fock = model.FockSpace(list(range(3)))
    H = sum((0.1 * i - 0.3) * fock.n(i) for i in range(3)) + 0.4 * fock.n(0) @ fock.n(1)
    ed = model.EDCore(H, fock, lambda b: b)
    grid = model.ImaginaryTimeGrid(5.0, 8)
    delta = 0.3 * model.bethe_gf(1.0, 5.0, grid)
    pairs = []
    for i in range(4):
        f, l = 1.0 + 0.1 * i, i % 3
        pairs.append(model.InteractionPair(f * fock.c_dag(l), fock.c(l), delta * (1 + 0.2 * i)))
        pairs.append(model.InteractionPair(f * fock.c(l), fock.c_dag(l), delta * (1 + 0.2 * ((i + 1) % 4))))
    return model.Expansion(ed, grid, pairs, [(-fock.c(0), fock.c_dag(0))])


F64, F32 = abi.QIW_PREC_FP64, abi.QIW_PREC_FP32
# walk: (its kernel, model, largest order of a step, of a correlator and of the self-energy, precision)
WALKS = {
    "flat": ("k_eval_flat_t", scaled_levels, 4, F64),
    "vector": ("k_eval_vec_t", lambda: many_pairs(3, particles), 2, F64),
    "vector, float32": ("k_eval_vec_t", lambda: many_pairs(3, particles), 2, F32),
    "matrix-core": ("k_eval_mfma_t", lambda: many_pairs(4, parity), 2, F32),
    "LDS block": ("k_eval_block", lambda: many_pairs(4, parity), 2, F64),
}
