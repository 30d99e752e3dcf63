"""Randomized solves at the edges of the launch that reduces a step's rows and draws the next
step's coordinates (k_step_reduce_finalize_rqmc), against the float64 oracle: coordinates in several
blocks of 512 samples, part of one, or one sample; rows of one and of several blocks of 256 elements;
reductions of 256 and of 1024 threads; at least two bold steps, so that drawn coordinates are used.
Tolerance 1e-10 relative, as for every float64 path; a deviation's error is bounded by 1e-10 of the
samples' scale."""
import numpy as np
import pytest

import oracle_lib as O
import qiw
from qiw import model
from test_gpu_bookkeeping import RTOL, rel, std_close

pytestmark = pytest.mark.gpu
MODELS = {"level": lambda n_tau: model.bethe_single_level(n_tau, 10.0),
          "two orbitals": lambda n_tau: model.kanamori(2, 2.0, 0.2, -1.0, 10.0, n_tau, 0.5),
          "three orbitals": lambda n_tau: model.kanamori(3, 3.0, 0.3, 0.0, 10.0, n_tau, 0.4)}


@pytest.mark.parametrize("which,n_tau,order,log2n,n_seqs", [
    ("level", 6, 3, 9, 3), ("level", 6, 3, 10, 3), ("level", 5, 2, 12, 2),  # one, two and eight blocks of coordinates
    ("level", 5, 2, 16, 2),                   # 1024 rows of two elements: 256 threads, 128 blocks of coordinates
    ("two orbitals", 5, 2, 6, 2),             # 1024 threads, 70 elements
    ("three orbitals", 5, 1, 0, 3),           # four blocks of elements, one sample
    ("three orbitals", 5, 1, 2, 9),           # sequences read from memory
    ("three orbitals", 4, 1, 4, 2)])          # 1024 threads
def test_sequences_drawn_beside_the_bookkeeping(which, n_tau, order, log2n, n_seqs):
    eg, ec = MODELS[which](n_tau), MODELS[which](n_tau)
    orders, N = range(0, order + 1), 2 ** log2n
    Po_g, Ps_g = qiw.inchworm(eg, eg.grid, orders, orders, N, rand_params=qiw.RandomizationParams(11, n_seqs, 0.0))
    P_c, Po_c, Ps_c = O.inchworm(ec, orders, orders, N, rand=(n_seqs, 1, 11, 0.0))
    assert rel(eg.P, P_c) < RTOL
    for o in orders:
        assert np.abs(Po_g[o] - Po_c[o]).max() < RTOL * np.abs(P_c).max()
        assert std_close(Ps_g[o], Ps_c[o], Po_c[o])
