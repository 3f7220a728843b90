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
