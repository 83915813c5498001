"""Host arrays in and out: what is uploaded comes back, element for element, at
sizes around the 1 MiB chunks the copies go in (part of one, exactly whole
ones, more than the four in flight), for fields, statuses and solver arrays."""
import numpy as np
import pytest

import incrmt_amd as ia

pytestmark = pytest.mark.gpu


# 131072 doubles are one chunk: (m+4)(n+4) below, at and above it, and above four
@pytest.mark.parametrize("m,n", [(8, 8), (252, 508), (256, 512), (124, 1020), (700, 796), (1020, 1020)])
def test_fields_come_back(m, n):
    f = ia.Fluid2D(m, n, visc=1e-2, rhof=1.0, x_prd=False, y_prd=False, ax=0.0, bx=1.0, ay=0.0, by=n / m)
    f.add_circle(0.5, 0.5 * n / m, 0.2 * min(1.0, n / m), 0.0, G=1.0, rhos=1.0)
    f.initialize()
    r = np.random.default_rng(m + n)
    for name in ("u", "p", "X"):
        a = r.standard_normal((n + 4, m + 4))
        f.set(name, a)
        assert np.array_equal(f.get(name), a), name
    s = r.integers(0, 8, (n + 4, m + 4)).astype(float)
    f.set("s", s)
    assert np.array_equal(f.get("s"), s)
    f.close()


@pytest.mark.parametrize("m,n", [(16, 8), (512, 256), (520, 260), (768, 1000)])
def test_solver_arrays(m, n):
    s = ia.MgSolver(ia.MG_MAC, m, n, 1.0, 1.0)
    x = np.random.default_rng(m).integers(-8, 9, (n, m)).astype(float)
    p = np.pad(x, 1, mode="edge")
    want = p[1:-1, 2:] + p[1:-1, :-2] + p[2:, 1:-1] + p[:-2, 1:-1] - 4 * x
    assert np.array_equal(s.apply(x).reshape(n, m), want)  # whole numbers: exact
    s.close()


def test_fixed_column_reads_as_zero():
    s = ia.MgSolver(ia.MG_FEM, 513, 512, 1.0, 1.0, y_prd=True, zpr=True)  # node column 512, two chunks
    y = s.apply(np.random.default_rng(1).standard_normal(513 * 512)).reshape(512, 513)
    assert np.all(y[:, 512] == 0) and np.all(y[:, :512] != 0)
    s.close()
