"""The single-workgroup tail of the V-cycle on systems that lie in it whole, or
nearly so: every factor size of the coarsest level, coarsest levels that are
swept (by one wavefront and by the workgroup), one and two groups of points a
thread. Solutions against a direct solve: the smallest eigenvalue over the
largest is above 1e-3 at these sizes, so a relative residual of 1e-11 bounds
the relative error by 1e-8."""
import numpy as np
import pytest

import incrmt_amd as ia
from tests import operators as ops

pytestmark = pytest.mark.gpu

MAC = [(2, 2), (3, 3), (4, 2), (4, 4), (8, 4), (5, 7), (12, 20), (32, 32), (36, 30), (44, 30), (64, 32)]
FEM = [(2, 2), (3, 3), (5, 3), (4, 4), (9, 9), (17, 5), (21, 41), (33, 33), (40, 24), (65, 33)]


@pytest.mark.parametrize("precision", [ia.PREC_FP64, ia.PREC_MIXED])
@pytest.mark.parametrize("kind,m,n", [("mac", *s) for s in MAC] + [("fem", *s) for s in FEM])
def test_tail_solves_match_direct(kind, m, n, precision):
    h = 1.0 / m
    if kind == "mac":
        irho = ops.mac_irho_from_rho(ops.blob_density(m, n, seed=3), m, n)
        s, A = ia.MgSolver(ia.MG_MAC, m, n, h, h), ops.mac_matrix(m, n, h, h, irho)
    else:
        irho = ops.fem_irho_from_rho(ops.blob_density(m - 1, n - 1, seed=3), m - 1, n - 1)
        s, A = ia.MgSolver(ia.MG_FEM, m, n, h, h), ops.fem_matrix(m, n, h, h, irho)
    s.set_irho(irho)
    b = np.random.default_rng(m + n).standard_normal(m * n)
    for _ in range(2):  # the second from the first's solution moved by a constant
        z, _, rr = s.solve(b, rel_tol=1e-11, max_cycles=400, precision=precision)
        assert rr <= 1e-11
        zd = ops.neumann_solve(A, b)
        assert np.linalg.norm((z - z.mean()) - zd) <= 1e-8 * np.linalg.norm(zd)
        s.solve(b + 0.1 * np.arange(m * n), rel_tol=1e-11, max_cycles=400, precision=precision, z=z + 2.0)
    s.close()
