"""Mixed-precision solves, where a cycle's end and the next one's residual are
one pass that leaves the iterate in the other buffer: V-cycles launched one by
one against the same replayed from the two graphs that the buffers need (the
same bits and cycle counts), and the residual that the pass reports against
the operator's matrix: both are formed in double from the same solution, whose
operator terms are at most about 1e4 times b, nine of them with a rounding
each, so the relative residuals agree to 1e-11. Sizes: within one block, odd
ones, and more points than the reduction has threads (several a thread)."""
import numpy as np
import pytest

import incrmt_amd as ia
from tests import operators as ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,m,n", [(ia.MG_MAC, *s) for s in ((2, 2), (9, 33), (64, 72), (400, 416), (1152, 128))]
                         + [(ia.MG_FEM, *s) for s in ((2, 2), (10, 34), (65, 73), (401, 417), (1153, 129))])
def test_one_pass(kind, m, n):
    h = 1.0 / m
    A = (ops.mac_matrix if kind == ia.MG_MAC else ops.fem_matrix)(m, n, h, h)
    s = [ia.MgSolver(kind, m, n, h, h) for _ in range(2)]
    for x, mode in zip(s, (ia.LAUNCH_DIRECT, ia.LAUNCH_GRAPH)):
        x.set_launch(mode)
    rng = np.random.default_rng(m)
    for tol in (1e-10, 1e-10, 1e-4):  # later solves run cycles ahead of their first check
        b = rng.standard_normal(m * n)
        z0 = rng.standard_normal(m * n)
        (za, ca, ra), (zb, cb, rb) = (x.solve(b, rel_tol=tol, max_cycles=60, precision=ia.PREC_MIXED, z=z0) for x in s)
        assert (ca, ra) == (cb, rb) and np.array_equal(za, zb), (ca, cb, ra, rb)
        b -= b.mean()
        assert abs(np.linalg.norm(b - A @ za) / np.linalg.norm(b) - ra) <= 1e-11
    for x in s:
        x.close()
