"""Resident solves in teams of different sizes: uneven batches with one
system that takes a large team, where each of the others takes a small one.

Iterates after 9 iterations differ from the streaming form's by the order of
the sums only, 1e-12 of the largest value as in tests/test_gpu_resident.py;
mixed solves end at the tolerance on the caller's FP64 operator.
"""
import numpy as np
import pytest

import eafp
import oracle
from eafp import systems
from test_gpu_resident import both, system

pytestmark = pytest.mark.gpu

LARGE = (40, 64, 40)
BATCHES = [[LARGE] + [(20, 30, 33)] * 11, [(9, 8, 64), (33, 17, 65), LARGE, (18, 36, 24), (5, 2, 33), LARGE],
           [LARGE] + [(12, 20, 16 + q) for q in range(40)]]


@pytest.mark.parametrize("batch", range(len(BATCHES)))
def test_fp64_iterates_in_uneven_teams(batch):
    syss = [system(s, q) for q, s in enumerate(BATCHES[batch])]
    print(f"case teams fp64 {batch}", flush=True)
    (st, phi), (st_s, phi_s) = both(syss, lambda b: b.solve_fp64(9, 1e-30))
    for s in range(len(syss)):
        assert st[s]["status"] == st_s[s]["status"] and st[s]["n_iter"] == st_s[s]["n_iter"]
        assert np.abs(phi[s] - phi_s[s]).max() <= 1e-12 * max(np.abs(phi_s[s]).max(), 1e-300)


@pytest.mark.parametrize("precond", [eafp._lib.PRECOND_JACOBI, eafp._lib.PRECOND_ZLINE])
@pytest.mark.parametrize("fmt", [eafp._lib.COEF_FP32, eafp._lib.COEF_BF16, eafp._lib.COEF_FP16])
def test_mixed_in_uneven_teams(precond, fmt):
    syss = [systems.make_system(2, 0, LARGE)] + [systems.make_system(3, s) for s in range(40)]
    print(f"case teams mixed fmt {fmt} precond {precond}", flush=True)
    with eafp.Batch.from_systems(syss) as b:
        st = b.solve_mixed(tol=1e-8, coef_format=fmt, precond=precond)
        for s, ps in enumerate(syss):
            assert st[s]["status"] == "converged" and st[s]["residual"] < 1e-8
            if s % 8 == 0:
                l2, _ = oracle.true_residual(ps, b.download(s))
                assert l2 < 1.2e-8
