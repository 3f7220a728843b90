"""Host arrays cross in pieces of at most 262,144 doubles, eight arrays gathered
one behind the other on the way in, p' by itself on the way back.

The copies change nothing: a batch uploaded from host arrays gives the same
doubles as one uploaded from device arrays, whatever the order of small and
large systems, and so does the drop-in, whose copies and solve run without a
wait between them.
"""
import numpy as np
import pytest

import eafp
from eafp.solver import COEF_NAMES
from hipbuf import HipBuffers
from test_gpu_layout import case

pytestmark = pytest.mark.gpu

# eight arrays are one full piece; one z-plane more; the smallest; one array is
# one full piece; one z-plane more; more pieces than there are slots
SHAPES = [(28, 28, 28), (28, 28, 29), (1, 1, 1), (60, 60, 60), (60, 60, 61), (100, 120, 84)]


def from_device(shape, ps, phi0, max_iter):
    buf = HipBuffers()
    with eafp.Batch([shape]) as B:
        B.upload_device(0, [buf.put(ps.padded(n)) for n in COEF_NAMES + ("Su",)],
                        None if phi0 is None else buf.put(phi0))
        B.solve_fp64(max_iter=max_iter, tol=1e-14)
        return B.download(0, np.zeros([n + 4 for n in shape], order="F"))


@pytest.mark.parametrize("shape", SHAPES)
def test_drop_in(shape):
    ps, phi0 = case(shape, 5)
    print(f"case host arrays shape={shape}", flush=True)
    ref = from_device(shape, ps, phi0, 3)
    for _ in range(3):     # the cached workspace's pinned memory is used again
        phi = phi0.copy(order="F")
        eafp.cg_3d_mpi(*[ps.padded(n) for n in COEF_NAMES], ps.Su, phi, eafp.Mesh(*shape), 3, 1e-14)
        assert np.array_equal(phi, ref)


@pytest.mark.parametrize("order", [(0, 1, 2, 3, 4), (4, 3, 2, 1, 0)])
def test_batch_of_small_and_large(order):
    shapes = [SHAPES[q] for q in order]
    print(f"case host arrays batch={shapes}", flush=True)
    cases = [case(s, 30 + q) for q, s in enumerate(shapes)]
    with eafp.Batch(shapes) as B, eafp.Batch(shapes) as D:
        buf = HipBuffers()
        for s, (ps, phi0) in enumerate(cases):
            p0 = phi0 if s % 2 else None
            B.upload(s, ps, p0)
            D.upload_device(s, [buf.put(ps.padded(n)) for n in COEF_NAMES + ("Su",)],
                            None if p0 is None else buf.put(p0))
        B.solve_fp64(max_iter=3, tol=1e-14)
        D.solve_fp64(max_iter=3, tol=1e-14)
        for s in range(len(shapes)):
            assert np.array_equal(B.download(s), D.download(s))
