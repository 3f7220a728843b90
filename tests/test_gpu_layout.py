"""The tiled transposes between the caller's padded arrays and the compact
layout, at the edges of their 32 x 32 tiles and with one and two theta planes.

One CG iterate of a diagonally dominant system with wall links, a non-zero
initial phi and non-zero halos reads every array that the pack moves, and the
halo products that it folds.  The iterate takes four sums over the cells,
each of terms of one sign or dominated by the diagonal: the two sides differ
by their order of summation, a few hundred roundings at most, and the bound
is the 1e-9 of the largest value that the other one-iterate tests have.
"""
import numpy as np
import pytest

import eafp
import oracle
from eafp.solver import COEF_NAMES
from fold_case import NAMES, FoldCase
from test_gpu_cg64 import check_halos

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (31, 2, 33), (32, 1, 32), (33, 3, 31), (64, 5, 65), (1, 7, 70), (97, 2, 1)]


def case(shape, seed):
    rng = np.random.default_rng(seed)
    padded = tuple(n + 4 for n in shape)
    arrs = {n: np.asfortranarray(rng.uniform(0.1, 1.0, padded)) for n in NAMES}
    arrs["aP"] = np.asfortranarray(1.0 + sum(arrs[n] for n in NAMES[:6]))
    return FoldCase(shape, arrs), np.asfortranarray(rng.normal(size=padded))


@pytest.mark.parametrize("shape", SHAPES)
def test_one_iterate_at_tile_edges(shape):
    ps, phi0 = case(shape, 11)
    print(f"case layout shape={shape}", flush=True)
    phi = phi0.copy(order="F")
    eafp.cg_3d_mpi(*[ps.padded(n) for n in COEF_NAMES], ps.Su, phi, eafp.Mesh(*shape), 1, 1e-14)
    ref, _, _, _ = oracle.cg(ps, phi0, max_iter=1, tol=1e-14)
    np.testing.assert_allclose(oracle.interior(phi), oracle.interior(ref), rtol=0,
                               atol=1e-9 * np.abs(oracle.interior(ref)).max())
    check_halos(phi, phi0, shape[1])


def test_every_system_of_a_batch_comes_back():
    """One launch writes the phi of every system: each system of a batch of
    different shapes gives the phi of a batch of its own."""
    cases = [case(s, 20 + q) for q, s in enumerate(SHAPES)]
    print("case layout batch", flush=True)
    with eafp.Batch(SHAPES) as B:
        for s, (ps, phi0) in enumerate(cases):
            B.upload(s, ps, phi0)
        B.solve_fp64(max_iter=1, tol=1e-14)
        for s, (ps, phi0) in enumerate(cases):
            phi = B.download(s)
            ref, _, _, _ = oracle.cg(ps, phi0, max_iter=1, tol=1e-14)
            np.testing.assert_allclose(oracle.interior(phi), oracle.interior(ref), rtol=0,
                                       atol=1e-9 * np.abs(oracle.interior(ref)).max())
            check_halos(phi, phi0, SHAPES[s][1])
