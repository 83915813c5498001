"""How often a solver captures its V-cycles: a graph is kept for each kind of
cycle and each choice of the iterate buffers that it uses (two; with the update
inside the cycle, of the FP64 and of the FP32 pair), so a handle's captures stop
growing whatever calls between its solves swap, and every solve gives what
directly launched cycles give."""
import numpy as np
import pytest

import incrmt_amd as ia

pytestmark = pytest.mark.gpu

# one sweep a launch (shape 3 for MAC, 1 for FEM): one sweep swaps one pair of buffers
KINDS = [(ia.MG_MAC, 128, 96, 3), (ia.MG_FEM, 129, 97, 1)]


def _pair(kind, m, n):
    s = [ia.MgSolver(kind, m, n, 1.0 / m, 1.3 / n) for _ in range(2)]
    for x, mode in zip(s, (ia.LAUNCH_GRAPH, ia.LAUNCH_DIRECT)):
        x.set_launch(mode)
    return s


def _solve(s, rng, precision, tol=1e-9):
    n = s[0].m * s[0].n
    b, z0 = rng.standard_normal(n), rng.standard_normal(n)
    a, d = (x.solve(b, rel_tol=tol, max_cycles=200, precision=precision, z=z0) for x in s)
    assert a[1:] == d[1:] and np.array_equal(a[0], d[0])
    return a[1]


@pytest.mark.parametrize("kind,m,n,shape", KINDS)
@pytest.mark.parametrize("precision", [ia.PREC_FP64, ia.PREC_MIXED])
def test_one_pair_swapped_between_mixed_solves(kind, m, n, shape, precision):
    s = _pair(kind, m, n)
    rng = np.random.default_rng(5)
    _solve(s, rng, ia.PREC_MIXED)
    assert s[0].captures == 2
    b, z = rng.standard_normal((2, m * n))
    y = [x.smooth(b, z, 1, shape, precision) for x in s]
    assert np.array_equal(*y)
    for _ in range(2):
        assert _solve(s, rng, ia.PREC_MIXED) > 2
    assert s[0].captures == 2
    for x in s:
        x.close()


@pytest.mark.parametrize("kind,m,n,shape", KINDS)
def test_precisions_in_turn(kind, m, n, shape):
    s = _pair(kind, m, n)
    rng = np.random.default_rng(6)
    cycles = set()
    for k in range(12):
        for x in s:
            x.set_krylov(k % 4 == 3)
        p = ia.PREC_MIXED if k % 2 else ia.PREC_FP64
        c = _solve(s, rng, p, 10.0 ** -rng.integers(4, 12))
        cycles.add(c % 2)
        if k % 3 == 0:
            y = [x.smooth(np.ones(m * n), np.arange(m * n) * 1e-3, 1, shape, p) for x in s]
            assert np.array_equal(*y)
    assert cycles == {0, 1}
    # FP64: two; mixed: two; Krylov: four at most
    assert s[0].captures <= 8 and s[1].captures == 0
    for x in s:
        x.close()
