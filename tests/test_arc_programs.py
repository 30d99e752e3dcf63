"""Arc programs (qinchworm.jl_amd/csrc/qiw_arcs.h): compiled with
g++ and run on the CPU word for word as the device kernels read them (every access
checked), against the plain sum over topologies and pair assignments, for every kind of group, orders
0 to 6, cut programs (fixed pairs), several wavefront counts and value sizes, narrow and wide
blocks.

Tolerance: both sides sum the same products of float64 factors of magnitude <= 1 in another
order; at most 4e3 diagrams of chains of 12 factors with blocks up to 20, so the difference
is below 4e3 * 12 * 20 * 2^-53 ~ 1e-10 of the largest term, and 1e-9 of the largest element
covers sums that cancel to a tenth of it."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "qinchworm.jl_amd", "csrc")
BOLD, BARE, CORR, SIGMA = range(4)


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path_factory.mktemp("arcs") / "arc_program")
    subprocess.run([gxx, "-O2", "-std=c++17", "-I", CSRC, os.path.join(HERE, "native", "arc_program_main.cpp"),
                    "-o", exe], check=True)
    return lambda *a: subprocess.run([exe] + [str(x) for x in a], capture_output=True, text=True, check=True).stdout


# kind, order, n_after, fixed pairs, wavefronts, LDS cap, bytes per value, modes, largest block
CASES = [(BOLD, 0, 0, 0, 1, 20000, 4, 2, 5), (BOLD, 1, 1, 0, 1, 20000, 4, 2, 5), (BOLD, 2, 1, 0, 1, 20000, 4, 2, 5),
         (BOLD, 2, 2, 0, 4, 20000, 4, 2, 8), (BOLD, 2, 3, 0, 1, 40000, 8, 3, 5), (BOLD, 3, 2, 0, 4, 60000, 4, 2, 20),
         (BOLD, 3, 3, 1, 4, 30000, 4, 2, 5), (BOLD, 3, 5, 2, 1, 40000, 8, 2, 7), (BOLD, 4, 4, 0, 16, 160000, 4, 2, 5),
         (BOLD, 4, 3, 1, 4, 40000, 8, 1, 5), (BOLD, 4, 7, 0, 8, 100000, 4, 2, 3), (BARE, 1, 2, 0, 1, 20000, 4, 2, 5),
         (BARE, 2, 4, 0, 4, 60000, 4, 2, 13), (BARE, 3, 6, 1, 4, 40000, 8, 2, 5), (CORR, 0, 0, 0, 1, 20000, 4, 2, 5),
         (CORR, 1, 1, 0, 1, 20000, 4, 2, 5), (CORR, 2, 1, 0, 2, 40000, 4, 3, 5), (CORR, 2, 2, 1, 4, 40000, 8, 2, 9),
         (CORR, 3, 4, 0, 8, 80000, 4, 2, 13), (SIGMA, 1, 1, 0, 1, 20000, 4, 2, 5), (SIGMA, 2, 1, 0, 4, 40000, 4, 3, 5),
         (SIGMA, 3, 1, 0, 4, 60000, 8, 2, 5)]
# the scalar programs (0 bytes per value): as few segments as fit, and cut into many
CASES += [(kind, order, na, cut, 1, 0, 0, modes, 1)
          for kind, order, na, modes in [(BOLD, 0, 0, 2), (BOLD, 1, 1, 2), (BOLD, 2, 2, 3), (BOLD, 3, 3, 3), (BOLD, 4, 4, 2),
                                         (BOLD, 5, 3, 1), (BOLD, 6, 6, 1), (BARE, 0, 0, 2), (BARE, 3, 6, 2), (CORR, 0, 0, 2),
                                         (CORR, 3, 2, 2), (CORR, 2, 3, 3), (SIGMA, 1, 1, 2), (SIGMA, 4, 1, 2)]
          for cut in (0, 1)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
def test_program_sums_the_diagrams(driver, case):
    for seed in (1, 2):
        out = driver(*case[:8], seed, case[8]).split()
        assert out[0] == "dev", out
        assert float(out[1]) < 1e-9
        assert out[3] == out[4]  # diagrams counted
        assert int(out[6]) <= (case[5] if case[6] else 300 * 512)


def test_states_beyond_the_lds(driver):
    """A group whose widest level exceeds the cap is refused, and fits when cut by the pair of
    its first arc."""
    assert driver(BOLD, 3, 3, 0, 4, 3000, 4, 3, 1).split() == ["rc", "2"]
    whole = driver(BOLD, 4, 4, 0, 4, 100000, 8, 2, 1).split()
    cut = driver(BOLD, 4, 4, 1, 4, int(whole[6]) - 1, 8, 2, 1).split()
    assert whole[0] == cut[0] == "dev" and float(cut[1]) < 1e-9


@pytest.mark.parametrize("kind,order", [(BOLD, 0), (BOLD, 1), (BARE, 0), (BARE, 2), (CORR, 0), (SIGMA, 1)])
def test_model_without_pairs(driver, kind, order):
    """No interaction pair: the propagator alone at order 0, no diagram above."""
    n_after = {BARE: 2 * order, SIGMA: 1}.get(kind, order)
    out = driver(kind, order, n_after, 0, 2, 20000, 8, 0, 1).split()
    assert out[0] == "dev" and float(out[1]) < 1e-9 and out[3] == out[4]
