"""Scarce memory on the GPU: what the resident solvers take on top of the
streaming ones never costs a call that fits without it.
"""
import pytest

import limits

pytestmark = pytest.mark.gpu

DEVICE = '''
shapes = [(20, 30, 33), (12, 24, 16), (9, 28, 35)]
syss = [systems.make_system(3, s, sh) for s, sh in enumerate(shapes)]

def solve(b, kind):
    if kind == "fp64":
        b.solve_fp64(40, 1e-30)
        b.set_tiling(1, 0)                            # more partial sums
        return b.solve_fp64(40, 1e-30)
    for fmt in (_lib.COEF_BF16, _lib.COEF_FP16):      # the second format's weights come on top of the first solve
        st = b.solve_mixed(tol=1e-8, coef_format=fmt, precond=_lib.PRECOND_ZLINE)
    return st

def take(kind, limit=-1, fail=-1):
    """(bytes, pieces) that the solve takes, with at most `limit` bytes or without
    the piece `fail`; None: out of memory."""
    with eafp.Batch.from_systems(syss) as b:
        used = shim.shim_used()
        shim.shim_limit(-1 if limit < 0 else used + limit)
        shim.shim_fail(fail)
        try:
            st = solve(b, kind)
        except eafp._lib.EafpError as e:
            assert e.rc == 2, e
            return None
        finally:
            shim.shim_limit(-1)
            calls = shim.shim_calls()
            shim.shim_fail(-1)
        assert all(s["status"] in ("converged", "max_iter") for s in st)
        return shim.shim_used() - used, calls

for kind in ("fp64", "mixed"):
    full, calls = take(kind)
    without = {c: take(kind, fail=c) for c in range(1, calls + 1)}      # a piece that the solve can do without
    need = min(t[0] for t in without.values() if t is not None)
    print("case", kind, full, calls, need, [c for c, t in without.items() if t is not None], flush=True)
    assert need < full
    assert take(kind, limit=need) is not None
    assert take(kind, limit=need - 1) is None
'''


def test_what_a_solve_can_do_without_costs_no_other_piece(tmp_path):
    limits.run(tmp_path, DEVICE)


PINNED = '''
ps = systems.make_system(2, 0, (20, 30, 33))
mesh = eafp.Mesh(*ps.shape)
F, cfg = fields.make_fields(*ps.shape, seed=3, masks=True)
tm = (35, 66, 49)                # large enough for overlapped passes
tps = systems.make_system(3, 0, tm)
names = ("aW", "aE", "aS", "aN", "aB", "aT", "aP", "Su")

def passes():
    coef = [np.array(ps.padded(n), order="F") for n in names]
    phi = np.zeros_like(coef[0], order="F")
    res, nit = eafp.cg_3d_mpi(*coef, phi, mesh, 30, 1e-30)
    out = {"cg": phi}
    assert nit == 30
    with eafp.Batch.from_systems([ps]) as b:
        st = b.solve_fp64(30, 1e-30)
        out["fp64"] = b.download(0)
        assert st[0]["n_iter"] == 30
        st = b.solve_mixed(tol=1e-10)
        assert st[0]["status"] == "converged"
        out["mixed"] = b.download(0)
    coef, res, flux = eafp.pp_assemble(F, cfg, mesh)
    out.update(coef, residual=np.array([res, flux]))
    t = [np.array(tps.padded(n), order="F") for n in names]
    f = np.asfortranarray(np.random.default_rng(1).normal(size=t[0].shape))
    eafp.tdma_3d_mpi(*t, f, eafp.Mesh(*tm), 2)
    out["tdma"] = f
    eafp.release()
    return out

with_it = passes()
shim.shim_pinned(8)              # the solvers' two counters, and nothing else
without = passes()
print("case", sorted(with_it), flush=True)
for n in with_it:
    if n in ("cg", "fp64", "mixed"):     # streaming instead of resident: the sums have another order
        tol = 1e-6 if n == "mixed" else 1e-12
        assert np.abs(with_it[n] - without[n]).max() <= tol * np.abs(with_it[n]).max(), n
    else:
        assert np.array_equal(with_it[n], without[n], equal_nan=True), n
'''


def test_without_pinned_memory(tmp_path):
    limits.run(tmp_path, PINNED)


SLOW = '''
ps = systems.make_system(2, 0, (35, 66, 49))
for solver in (eafp.Batch.SOLVER_FP64, eafp.Batch.SOLVER_MIXED_ZLINE):
    with eafp.Batch.from_systems([ps]) as b:
        shim.shim_slow(-1)
        quiet = b.autotune(solver, _lib.COEF_BF16, reps=2)
        calls = shim.shim_times()
        shim.shim_slow(calls)        # the last launch that is timed
        held_up = b.autotune(solver, _lib.COEF_BF16, reps=2)
        assert shim.shim_times() == calls
        shim.shim_slow(-1)
        print("case slow", solver, calls, quiet, held_up, flush=True)
        # the streaming kernels take twice as long on this mesh
        assert held_up["ms_per_iter"] < 1.5 * quiet["ms_per_iter"]
        assert b.resident(solver)["in_use"]
'''


def test_one_launch_held_up_does_not_decide(tmp_path):
    limits.run(tmp_path, SLOW)
