"""A system that no solver can do anything with does not reach the one before it
in a batch: rows that end inside a lane's four cells are read past their end,
which is where the next system begins when the cells are a multiple of 32."""
import numpy as np
import pytest

import eafp
from eafp import _lib, systems

pytestmark = pytest.mark.gpu


def solve(syss, fmt):
    with eafp.Batch.from_systems(syss) as b:
        st = b.solve_mixed(tol=1e-9, max_steps=100, coef_format=fmt, precond=_lib.PRECOND_ZLINE)
        return st[0], b.download(0)


@pytest.mark.parametrize("shape", [(8, 24, 34), (16, 24, 33), (8, 24, 84), (8, 16, 37)])
@pytest.mark.parametrize("fmt", [_lib.COEF_FP32, _lib.COEF_BF16, _lib.COEF_FP16])
def test_the_system_before_a_hopeless_one(shape, fmt):
    assert np.prod(shape) % 32 == 0
    good, fine, bad = (systems.make_system(2, s, shape) for s in range(3))
    for k in range(8):      # diagonals far below the links: factors beyond FP16 in the first row
        links = sum(bad.coef[n][2, 2, 2 + k] for n in ("aW", "aE", "aS", "aN", "aB", "aT"))
        bad.coef["aP"][2, 2, 2 + k] = (1e-6 if k % 2 == 0 else 1.0) * max(links, 1.0)
    print(f"case neighbour {shape} {fmt}", flush=True)
    st, phi = solve([good, bad], fmt)
    st_f, phi_f = solve([good, fine], fmt)
    print(st["status"], st["n_refine"], st_f["status"], st_f["n_refine"], flush=True)
    assert st["status"] == st_f["status"] == "converged"
    assert st["n_iter"] == st_f["n_iter"] and np.array_equal(phi, phi_f)
