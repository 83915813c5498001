"""The one-pass ends of mixed cycles (update, next residual, its rounding and
its norms in one kernel) against the separate passes, which a simulation takes
when a network is attached to its solvers, bit for bit: fields, cycle counts
and reported residuals over steps whose solves start from the previous solution
or a quadratic extrapolation (there run-ahead cycles go unchecked), for MAC and
FEM, walled and with a zero-pressure edge, launched one by one and replayed.
The network is attached by asking for the learned start and then dropped in
favour of the start under test, before any solve. Sizes: odd factors, and more
points than the reduction has threads (several a thread)."""
import numpy as np
import pytest

import incrmt_amd as ia

pytestmark = pytest.mark.gpu


def _spin(m):
    return ia.simple_spin(m, rel_tol=1e-10, precision=ia.PREC_MIXED)


def _outflow(m, n):
    f = ia.Fluid2D(m, n, visc=1e-2, rhof=1.0, ax=-1.0, bx=-1.0 + 2.0 * m / n, ay=-1.0, by=1.0)
    f.add_circle(0.1, -0.05, 0.3, 0.0, G=2.0, rhos=1.5)
    f.set_horizontal_flow(1.0)
    f.set_solver(rel_tol=1e-10, precision=ia.PREC_MIXED)
    f.initialize(0.8, 0.4, 0.8)
    return f


CASES = {"spin_56": lambda: _spin(56), "spin_72": lambda: _spin(72), "spin_384": lambda: _spin(384),
         "outflow_64": lambda: _outflow(64, 48), "outflow_512": lambda: _outflow(512, 384)}


@pytest.mark.parametrize("case", sorted(CASES))
@pytest.mark.parametrize("guess", [ia.GUESS_PREVIOUS, ia.GUESS_QUADRATIC])
@pytest.mark.parametrize("mode", [ia.LAUNCH_DIRECT, ia.LAUNCH_GRAPH])
def test_one_pass_equals_separate_passes(case, guess, mode):
    one, separate = CASES[case](), CASES[case]()
    separate.set_guess(ia.GUESS_LEARNED)
    for f in (one, separate):
        f.set_guess(guess)
        f.set_launch(mode)
    names = ("mac_cycles", "fem_cycles", "mac_rel_res", "fem_rel_res")
    cycles = 0
    for _ in range(6):
        for f in (one, separate):
            f.step_forward(one.dt_reg)
        a, b = one.stats(), separate.stats()
        assert [a[k] for k in names] == [b[k] for k in names]
        cycles += a["mac_cycles"] + a["fem_cycles"]
        for name in ("u", "v", "p"):
            assert np.array_equal(one.get(name), separate.get(name)), name
    assert cycles > 24
    for kind in (ia.MG_MAC, ia.MG_FEM):
        assert separate.guess_stats(kind)["learned_solves"] == 0
    one.close()
    separate.close()
