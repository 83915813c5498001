"""Mixed-precision solves with cycles launched one by one, where a cycle's end
and the next one's residual are one pass, against the same solves replayed from
captured graphs, where they are two passes. Stated bar: the same bits and
cycle counts, since every sum keeps its order. Sizes: within one block, odd
ones, and more points than the reduction has threads (several a thread)."""
import numpy as np
import pytest

import incrmt_amd as ia

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,m,n", [(ia.MG_MAC, *s) for s in ((2, 2), (9, 33), (64, 72), (400, 416), (1152, 128))]
                         + [(ia.MG_FEM, *s) for s in ((2, 2), (10, 34), (65, 73), (401, 417), (1153, 129))])
def test_one_pass_equals_two(kind, m, n):
    s = [ia.MgSolver(kind, m, n, 1.0 / m, 1.0 / m) for _ in range(2)]
    for x, mode in zip(s, (ia.LAUNCH_DIRECT, ia.LAUNCH_GRAPH)):
        x.set_launch(mode)
    rng = np.random.default_rng(m)
    for tol in (1e-10, 1e-10, 1e-4):  # later solves run cycles ahead of their first check
        b = rng.standard_normal(m * n)
        z0 = rng.standard_normal(m * n)
        (za, ca, ra), (zb, cb, rb) = (x.solve(b, rel_tol=tol, max_cycles=60, precision=ia.PREC_MIXED, z=z0) for x in s)
        assert (ca, ra) == (cb, rb) and np.array_equal(za, zb), (ca, cb, ra, rb)
    for x in s:
        x.close()
