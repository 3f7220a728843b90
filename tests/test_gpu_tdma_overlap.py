"""Overlapped line-TDMA sweeps (parts of the passes side by side) against
the oracle, bit for bit: meshes whose portions are whole tiles, one cell more
and one less, and batches in which some systems have empty portions."""
import pytest

import eafp
import oracle
from test_gpu_tdma import NAMES, assert_bitwise, random_system

pytestmark = pytest.mark.gpu

BATCHES = [[(40, 50, 41)], [(17, 200, 33)], [(64, 65, 64)], [(33, 70, 49)], [(7, 30, 600)], [(120, 128, 3)],
           [(40, 50, 41), (5, 7, 6), (1, 3, 2), (16, 9, 48), (2, 70, 3)]]


def solve(shapes, n_sweep, huge):
    sys_, wants = [], []
    for q, shape in enumerate(shapes):
        coef, phi0 = random_system(shape, 900 + sum(shape) + q, huge=(huge == q))
        wants.append(oracle.tdma_3d(coef, phi0, shape, n_sweep))
        sys_.append(dict(coef, phi=phi0.copy(order="F")))
    eafp.tdma_batch(sys_, [eafp.Mesh(*s) for s in shapes], n_sweep)
    for q, shape in enumerate(shapes):
        assert_bitwise(sys_[q]["phi"], wants[q], f"system {q} {shape}")


@pytest.mark.parametrize("shapes", BATCHES, ids=str)
def test_overlapped_sweeps_match_oracle_bitwise(shapes):
    print(f"case tdma overlap {shapes}", flush=True)
    solve(shapes, 3, None)


def test_a_pivot_out_of_band_keeps_the_passes_in_turn():
    """One system's pivots leave the chain kernel's band: its passes run on the
    other kernel, whole, so the call takes the passes one after another."""
    print("case tdma overlap with pivots out of band", flush=True)
    solve([(40, 50, 41), (12, 24, 16)], 2, 1)
