"""The resident solvers' paths that a result alone does not tell apart: which
form a solve took, and what follows a launch that is given up, sum numbers
that begin again, and solves of several threads at once.
"""
import threading
import time

import numpy as np
import pytest

import eafp
from eafp import _lib, systems
from test_gpu_resident import BIG, ROWS, system
from test_gpu_teams import BATCHES, LARGE

pytestmark = pytest.mark.gpu

FP64, MIXED = 0, 1
ZLINE = _lib.PRECOND_ZLINE


def solve(b, solver, n_iter=40):
    if solver == FP64:
        return b.solve_fp64(n_iter, 1e-30)
    return b.solve_mixed(tol=1e-9, coef_format=_lib.COEF_BF16, precond=ZLINE)


def outcome(b, solver, **kw):
    st = solve(b, solver, **kw)
    return [b.download(s) for s in range(len(b))] + [np.array([(s["n_iter"], s["residual"]) for s in st])]


def same(a, b):
    return all(np.array_equal(x, y, equal_nan=True) for x, y in zip(a, b))


def streamed(syss, solver):
    with eafp.Batch.from_systems(syss) as b:
        i = b.info()
        b.set_tiling(i["tile_cells"] // 256, i["grid"])
        assert not solve(b, solver)[0]["n_iter"] == 0
        r = b.resident(solver)
        assert r["launches"] == 0 and not r["in_use"]
        return outcome(b, solver)


@pytest.mark.parametrize("shape", ROWS + BIG)
@pytest.mark.parametrize("precond", [_lib.PRECOND_JACOBI, _lib.PRECOND_ZLINE])
@pytest.mark.parametrize("fmt", [_lib.COEF_FP32, _lib.COEF_BF16, _lib.COEF_FP16])
def test_which_form_a_mixed_solve_takes(shape, precond, fmt):
    """On chip up to the longest row that a wave holds: every step is a resident
    launch, unless the system is set aside."""
    with eafp.Batch.from_systems([system(shape, 3)]) as b:
        c0 = eafp.counters()["graph_launches"]
        st = b.solve_mixed(tol=1e-9, coef_format=fmt, precond=precond)[0]
        steps = eafp.counters()["graph_launches"] - c0
        r = b.resident(MIXED)
    print(f"case form {shape} fmt {fmt} precond {precond}: {r} {st['status']} {st['n_refine']}", flush=True)
    if shape[2] > 512:
        assert r["work_groups"] == 0 and r["launches"] == 0
        return
    assert r["work_groups"] > 0 and r["in_use"] and r["given_up"] == 0
    if r["set_aside"]:
        assert 0 < r["launches"] < steps
    else:
        assert r["launches"] == steps >= st["n_refine"]


def test_a_diverging_system_is_set_aside():
    with eafp.Batch.from_systems([systems.make_system(4, 257 * 948717418, (21, 77, 8))]) as b:
        b.solve_mixed(tol=1e-9, max_steps=60, coef_format=_lib.COEF_FP16, precond=_lib.PRECOND_JACOBI)
        assert b.resident(MIXED)["set_aside"] == 1


@pytest.mark.parametrize("solver", [FP64, MIXED])
@pytest.mark.parametrize("batch", ["one large", "one large, forty uneven"])
def test_uneven_batches_take_teams_of_different_sizes(solver, batch):
    syss = [system(s, q) for q, s in enumerate(BATCHES[0])] if batch == "one large" else \
        [systems.make_system(2, 0, LARGE)] + [systems.make_system(3, s) for s in range(40)]
    with eafp.Batch.from_systems(syss) as b:
        solve(b, solver)
        r = b.resident(solver)
    print("case teams", solver, batch, r, flush=True)
    assert r["launches"] > 0 and r["given_up"] == 0 and r["teams"] > 1 and r["team_size"] == 0


@pytest.mark.parametrize("solver", [FP64, MIXED])
def test_a_launch_that_is_given_up(solver):
    """A launch that waits for a work-group too many gives up; the solve and the
    next ones are the streaming kernels', until the pause is over."""
    syss = [systems.make_system(2, 0, (20, 30, 33)), systems.make_system(2, 1, (9, 28, 35))]
    print("case given up", solver, flush=True)
    stream = streamed(syss, solver)
    with eafp.Batch.from_systems(syss) as b:
        first = outcome(b, solver)
        n = b.resident(solver)["launches"]
        b.disturb(solver, _lib.DISTURB_ABSENT, 1)
        assert same(outcome(b, solver), stream)
        r = b.resident(solver)
        assert r["given_up"] == 1 and not r["in_use"] and r["launches"] > n
        b.disturb(solver, _lib.DISTURB_ABSENT, 0)
        assert same(outcome(b, solver), stream)              # not tried again at once
        assert b.resident(solver)["launches"] == r["launches"]
        b.disturb(solver, _lib.DISTURB_PAUSE, 1)
        time.sleep(1.1)
        assert b.resident(solver)["in_use"]
        assert same(outcome(b, solver), first)               # on chip again
        assert b.resident(solver)["given_up"] == 1 and b.resident(solver)["launches"] > r["launches"]


@pytest.mark.parametrize("solver,shapes,back", [
    (FP64, [(60, 120, 84)], 2050 + 100),          # the second launch of 1306 iterations begins again
    (MIXED, [(35, 66, 49)], 66 * 5),              # steps of 32 iterations
    (MIXED, [LARGE] + [(12, 20, 16)] * 300, 66 * 40),
])
def test_sum_numbers_that_begin_again(solver, shapes, back):
    syss = [systems.make_system(2, s % 7, sh) for s, sh in enumerate(shapes)]
    print("case tags", solver, shapes[0], flush=True)

    def full(b):
        return [b.solve_fp64(tol=1e-8)] if solver == FP64 else [solve(b, solver)]

    with eafp.Batch.from_systems(syss) as b:
        a = full(b)
        phi = [b.download(s) for s in range(len(b))]
        b.disturb(solver, _lib.DISTURB_TAG, 0xF0000000 - back)
        again = full(b)
        assert same(phi, [b.download(s) for s in range(len(b))])
        assert [x["n_iter"] for x in a[0]] == [x["n_iter"] for x in again[0]]
        assert b.resident(solver)["given_up"] == 0
        b.disturb(solver, _lib.DISTURB_TAG, 0x10000000)      # accepted: the numbers have begun again


def test_two_threads_with_a_batch_each():
    """Together the launches need more than the chip: they take turns."""
    jobs = [(FP64, [systems.make_system(2, 0, (60, 120, 84))]),
            (MIXED, [systems.make_system(2, s, (40, 64, 40)) for s in range(6)]),
            (FP64, [systems.make_system(3, s) for s in range(12)])]
    batches = [eafp.Batch.from_systems(syss) for _, syss in jobs]
    alone = [outcome(b, solver, n_iter=300) for b, (solver, _) in zip(batches, jobs)]
    bad = []

    def work(q):
        for _ in range(5):
            if not same(outcome(batches[q], jobs[q][0], n_iter=300), alone[q]):
                bad.append(q)

    print("case threads", flush=True)
    threads = [threading.Thread(target=work, args=(q,)) for q in range(len(jobs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    used = [b.resident(solver) for b, (solver, _) in zip(batches, jobs)]
    for b in batches:
        b.close()
    assert not bad
    assert all(r["given_up"] == 0 and r["launches"] > 0 for r in used)
