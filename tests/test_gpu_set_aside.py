"""A diverging system among others of a mixed batch on the GPU: it alone begins
again with the streaming kernels.  The others' results are those of a batch
without it, and its own is the streaming batch's, both bit for bit.
"""
import numpy as np
import pytest

import eafp
from eafp import _lib, systems

pytestmark = pytest.mark.gpu

HEALTHY = [(2, 0, (35, 66, 49)), (3, 1, (18, 36, 24)), (2, 2, (33, 17, 65))]
# systems that FP16 weights round into ones that refinement does not solve
DIVERGING = {_lib.PRECOND_JACOBI: [(4, 257 * 948717418, (21, 77, 8)), (4, 257 * 713431381, (26, 18, 60))],
             _lib.PRECOND_ZLINE: [(4, 257 * 1041356065, (21, 85, 21)), (4, 257 * 796802793, (24, 85, 11))]}


def solve(syss, precond, streaming=False):
    with eafp.Batch.from_systems(syss) as b:
        if streaming:
            i = b.info()
            b.set_tiling(i["tile_cells"] // 256, i["grid"])
        st = b.solve_mixed(tol=1e-9, max_steps=120, coef_format=_lib.COEF_FP16, precond=precond)
        return st, [b.download(s) for s in range(len(syss))]


@pytest.mark.parametrize("precond", sorted(DIVERGING))
@pytest.mark.parametrize("place", [0, 2])
def test_only_the_diverging_systems_begin_again(precond, place):
    print(f"case set aside precond {precond} place {place}", flush=True)
    far = DIVERGING[precond]
    bad = {place: far[0], 4: far[1]}
    rest = [systems.make_system(*h) for h in HEALTHY]
    order = [None if q in bad else rest.pop(0) for q in range(5)]
    with_bad = [systems.make_system(*bad[q]) if p is None else p for q, p in enumerate(order)]
    without = [systems.make_system(2, 5, bad[q][2]) if p is None else p for q, p in enumerate(order)]
    c0 = eafp.counters()["graph_launches"]
    st, phi = solve(with_bad, precond)
    launches = eafp.counters()["graph_launches"] - c0
    st_w, phi_w = solve(without, precond)
    st_s, phi_s = solve(with_bad, precond, streaming=True)
    for q in range(5):
        print(q, st[q]["status"], st[q]["n_refine"], st_w[q]["n_refine"], st_s[q]["n_refine"], flush=True)
        if q in bad:
            assert st[q]["status"] == st_s[q]["status"] == "max_iter"
            assert np.array_equal(phi[q], phi_s[q]) and st[q]["n_iter"] == st_s[q]["n_iter"]
            assert st[q]["residual"] == st_s[q]["residual"]
        else:
            assert st[q]["status"] == "converged"
            assert np.array_equal(phi[q], phi_w[q]) and st[q]["n_iter"] == st_w[q]["n_iter"]
    # the others' steps on chip, one launch each, then every step of the two
    assert launches >= max(st[q]["n_refine"] for q in range(5) if q not in bad) + 120


# systems that converge after their residual was up to 373 times its least
UNSTEADY = [((71, 15, 86), 297172762, _lib.COEF_FP32, _lib.PRECOND_ZLINE),
            ((11, 78, 71), 1045996112, _lib.COEF_FP32, _lib.PRECOND_JACOBI),
            ((13, 36, 47), 824138931, _lib.COEF_BF16, _lib.PRECOND_JACOBI),
            ((15, 24, 23), 172062608, _lib.COEF_BF16, _lib.PRECOND_ZLINE)]


@pytest.mark.parametrize("shape,seed,fmt,precond", UNSTEADY)
def test_an_unsteady_system_stays_on_chip(shape, seed, fmt, precond):
    print(f"case unsteady {shape} fmt {fmt} precond {precond}", flush=True)
    with eafp.Batch.from_systems([systems.make_system(4, 257 * seed, shape)]) as b:
        c0 = eafp.counters()["graph_launches"]
        st = b.solve_mixed(tol=1e-10, coef_format=fmt, precond=precond)[0]
        launches = eafp.counters()["graph_launches"] - c0
    assert st["status"] == "converged"
    assert launches <= st["n_refine"] + 2       # one per refinement step: nothing solved again
