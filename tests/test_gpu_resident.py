"""The resident solvers (systems kept on chip) on the GPU, at the sizes where
their division of a system changes form: one cell per axis, an uncut and a cut
theta ring, rows longer than a work-group, one member and many, the largest
number of cells per thread, and solves that a second launch takes up.

Default batches take the resident form; a launch shape asked for
(set_tiling) takes the streaming kernels.  Iterates after a few iterations
differ between the two only by the order of the sums, a few units of the
last place each: 1e-12 of the largest value, as the oracle comparison of
tests/test_gpu_cg64.py has it.
"""
import numpy as np
import pytest

import eafp
import oracle
from eafp import _lib, systems

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (1, 1, 5), (1, 3, 700), (3, 1, 7), (2, 2, 1), (5, 2, 33), (7, 50, 20), (9, 8, 64), (33, 17, 65),
          (40, 64, 3), (18, 36, 24), (35, 66, 50), (60, 119, 83)]


def system(shape, index=0):
    if min(shape[0], shape[1], shape[2]) > 4:
        return systems.make_system(2, index, shape)
    # the generator's masks leave no cell on the thinnest meshes: a random
    # diagonally dominant system instead
    rng = np.random.default_rng([index, *shape])
    g = systems.make_geometry(*shape)
    ps = systems.assemble(g, np.ones(shape, dtype=bool), np.full(shape, 1.2), tuple(rng.uniform(0.5, 2.0, shape)
                                                                                   for _ in range(3)), rng)
    ps.coef["aP"][2:-2, 2:-2, 2:-2] += rng.uniform(0.01, 0.1, shape) * ps.coef["aP"][2:-2, 2:-2, 2:-2].max()
    ps.Su[2:-2, 2:-2, 2:-2] = rng.normal(size=shape)
    return ps


def both(syss, solve):
    out = []
    for stream in (False, True):
        with eafp.Batch.from_systems(syss) as b:
            if stream:
                b.set_tiling(2, 0)
            st = solve(b)
            out.append((st, [b.download(s) for s in range(len(syss))]))
    return out


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("max_iter", [0, 1, 2, 9])
def test_fp64_iterates(shape, max_iter):
    ps = system(shape)
    (st, phi), (st_s, phi_s) = both([ps], lambda b: b.solve_fp64(max_iter, 1e-30))
    ref, _, nit, _ = oracle.cg(ps, max_iter=max_iter, tol=1e-30)
    print(f"case fp64 {shape} {max_iter}: {st[0]['status']} {st_s[0]['status']} n {st[0]['n_iter']} {nit}", flush=True)
    assert st[0]["status"] == st_s[0]["status"] and st[0]["n_iter"] == st_s[0]["n_iter"] == nit
    scale = max(np.abs(ref).max(), 1e-300)
    assert np.abs(phi[0] - phi_s[0]).max() <= 1e-12 * scale
    assert np.abs(oracle.interior(phi[0]) - oracle.interior(ref)).max() <= 1e-12 * scale


def test_fp64_past_one_launch():
    """1306 iterations to 1e-8: the second launch goes on where the first one
    stopped."""
    ps = systems.make_system(2)
    (st, phi), (st_s, phi_s) = both([ps], lambda b: b.solve_fp64(tol=1e-8))
    assert st[0]["status"] == "converged" and st[0]["n_iter"] > 1024
    assert abs(st[0]["n_iter"] - st_s[0]["n_iter"]) <= 2
    assert oracle.gauge_error(oracle.interior(phi[0]), oracle.interior(phi_s[0]), ps.labels, ps.ncomp) < 1e-9


def test_fp64_uneven_batch_with_failures():
    """Teams with several systems each; a zero right-hand side, a NaN and a
    thin mesh among them; repeats are bit-identical."""
    syss = [systems.make_system(3, s) for s in range(20)] + [system((1, 3, 700))]
    zero, nan = systems.make_system(1, 1), systems.make_system(1, 2)
    zero.Su[:] = 0.0
    nan.Su[6, 7, 8] = np.nan
    syss += [zero, nan]
    with eafp.Batch.from_systems(syss) as b:
        st = b.solve_fp64(1500, 1e-8)
        phi = [b.download(s) for s in range(len(syss))]
        again = b.solve_fp64(1500, 1e-8)
        for s in range(len(syss)):
            np.testing.assert_array_equal(b.download(s), phi[s])
            assert again[s]["n_iter"] == st[s]["n_iter"]
    assert st[-2]["status"] == "zero_rhs" and st[-2]["n_iter"] == 0
    assert st[-1]["status"] == "max_iter" and st[-1]["n_iter"] == 1500 and np.isnan(st[-1]["residual"])
    for s in (0, 7, 19):
        ref, _, nit, _ = oracle.cg(syss[s])
        assert st[s]["status"] == "converged" and abs(st[s]["n_iter"] - nit) <= 2
        assert oracle.gauge_error(oracle.interior(phi[s]), oracle.interior(ref), syss[s].labels, syss[s].ncomp) < 1e-9


# z-rows: one cell to one more than a wave holds with one quad per lane, and
# with two; the last one streams
ROWS = [(5, 7, 1), (4, 6, 3), (6, 5, 4), (3, 9, 63), (4, 6, 64), (5, 4, 65), (16, 24, 84), (4, 5, 129), (3, 8, 168),
        (3, 4, 255), (2, 3, 257), (2, 3, 512), (2, 2, 513)]
BIG = [(18, 36, 24), (35, 66, 49), (60, 120, 84), (61, 119, 83)]


def true_residual(ps, phi):
    l2, _ = oracle.true_residual(ps, phi)
    return l2


@pytest.mark.parametrize("shape", ROWS + BIG)
@pytest.mark.parametrize("precond", [eafp._lib.PRECOND_JACOBI, eafp._lib.PRECOND_ZLINE])
@pytest.mark.parametrize("fmt", [eafp._lib.COEF_FP32, eafp._lib.COEF_BF16, eafp._lib.COEF_FP16])
def test_mixed_matches_streaming(shape, precond, fmt):
    """Both forms end the same way.  Where they reach the tolerance, they do
    so on the caller's FP64 operator and with the same solution.  (The inner
    counts are not compared: the streaming forms' own differ by up to two
    refinement steps with the order of their sums.  On meshes that the inner CG solves in
    fewer iterations than a refinement step has, the kept search direction
    can stall the refinement with rounded weights, in both forms alike.)"""
    ps = system(shape, 3)
    c0 = eafp.counters()["graph_launches"]
    (st, phi), (st_s, phi_s) = both([ps], lambda b: b.solve_mixed(tol=1e-9, coef_format=fmt, precond=precond))
    launches = eafp.counters()["graph_launches"] - c0
    print(f"case mixed {shape} fmt {fmt} precond {precond}: inner {st[0]['n_iter']} {st_s[0]['n_iter']}", flush=True)
    assert st[0]["status"] == st_s[0]["status"]
    if st[0]["status"] != "converged":
        assert min(shape) < 18 and 0.1 < st[0]["residual"] / st_s[0]["residual"] < 10.0
        return
    for s, x in ((st[0], phi[0]), (st_s[0], phi_s[0])):
        assert s["residual"] < 1e-9
        assert true_residual(ps, x) < 1.2e-9
    assert launches <= st[0]["n_refine"] + st_s[0]["n_refine"] + 4    # no launch was given up and solved again
    assert oracle.gauge_error(oracle.interior(phi[0]), oracle.interior(phi_s[0]), ps.labels, ps.ncomp) < 1e-6


@pytest.mark.parametrize("precond", [eafp._lib.PRECOND_JACOBI, eafp._lib.PRECOND_ZLINE])
def test_mixed_uneven_batch_with_failures(precond):
    """Teams with several systems each; a zero right-hand side and a NaN among
    them; restart mode; repeats are bit-identical."""
    syss = [systems.make_system(3, s) for s in range(40)] + [system((6, 5, 4))]
    zero, nan = systems.make_system(1, 1), systems.make_system(1, 2)
    zero.Su[:] = 0.0
    nan.Su[6, 7, 8] = np.nan
    syss += [zero, nan]
    for restart in (False, True):
        with eafp.Batch.from_systems(syss) as b:
            st = b.solve_mixed(tol=1e-8, max_steps=60, coef_format=eafp._lib.COEF_BF16, precond=precond, restart=restart)
            phi = [b.download(s) for s in range(len(syss))]
            again = b.solve_mixed(tol=1e-8, max_steps=60, coef_format=eafp._lib.COEF_BF16, precond=precond,
                                  restart=restart)
            for s in range(len(syss)):
                np.testing.assert_array_equal(b.download(s), phi[s])
                assert again[s]["n_iter"] == st[s]["n_iter"]
            b.set_tiling(2, 0)
            streamed = b.solve_mixed(tol=1e-8, max_steps=60, coef_format=eafp._lib.COEF_BF16, precond=precond,
                                     restart=restart)
        print(f"case mixed batch precond {precond} restart {restart}: {[x['status'] for x in st]}", flush=True)
        assert [x["status"] for x in st] == [x["status"] for x in streamed]
        assert st[-2]["status"] == "zero_rhs"
        assert st[-1]["status"] == "max_iter" and np.isnan(st[-1]["residual"])
        for s in range(41):
            if st[s]["status"] == "converged":
                assert true_residual(syss[s], phi[s]) < 1.2e-8


def test_fp64_default_does_not_stream():
    """A default FP64 solve launches no graph of the streaming kernels."""
    ps = systems.make_system(1)
    c0 = eafp.counters()["graph_launches"]
    with eafp.Batch.from_systems([ps]) as b:
        b.solve_fp64(tol=1e-8)
        assert eafp.counters()["graph_launches"] == c0
        b.set_tiling(2, 0)
        b.solve_fp64(tol=1e-8)
        assert eafp.counters()["graph_launches"] > c0


@pytest.mark.parametrize("shape,seed,fmt,precond", [
    ((9, 28, 68), 1, "COEF_FP16", "PRECOND_ZLINE"),
    ((27, 31, 34), 2, "COEF_FP16", "PRECOND_ZLINE"),
    ((10, 85, 9), 3, "COEF_FP16", "PRECOND_JACOBI"),
    ((16, 52, 9), 4, "COEF_FP16", "PRECOND_JACOBI"),
])
def test_a_solve_that_diverges_is_the_streaming_one(shape, seed, fmt, precond):
    """16-bit weights can round a system into one that refinement does not
    solve.  What such a solve leaves is the streaming kernels' result, bit for
    bit; one that converges agrees with theirs to the tolerance."""
    ps = systems.make_system(4, seed, shape)
    print(f"case diverging shape={shape} seed={seed} {fmt} {precond}", flush=True)
    out = []
    for streaming in (False, True):
        with eafp.Batch([shape]) as B:
            if streaming:
                i = B.info()
                B.set_tiling(i["tile_cells"] // 256, i["grid"])
            B.upload(0, ps)
            st = B.solve_mixed(tol=1e-10, max_steps=600, coef_format=getattr(_lib, fmt),
                               precond=getattr(_lib, precond))[0]
            out.append((st, B.download(0)))
    (a, pa), (b, pb) = out
    print(a["status"], a["n_refine"], a["residual"], b["status"], b["n_refine"], b["residual"], flush=True)
    assert a["status"] == b["status"]
    if b["status"] == "converged":
        assert np.abs(pa - pb).max() <= 1e-6 * np.abs(pb).max()
    else:
        assert np.array_equal(pa, pb) and a["n_iter"] == b["n_iter"]
