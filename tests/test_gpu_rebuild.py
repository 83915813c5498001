"""The band rebuild's scan, dilation and finalisation where their row groups and
votes end: remainders of a thread's rows and of a wavefront's columns, and
dilation radii just inside and past one and two wavefronts of columns. Bit for
bit against the oracle, as in every other band comparison."""
import numpy as np
import pytest

import incrmt_amd as ia
from tests import oracle_lib as ol

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n", [(8, 8), (63, 17), (64, 16), (65, 19), (130, 34), (261, 50)])
@pytest.mark.parametrize("cells", [2.0, 60.0, 61.0, 62.0, 126.0])
def test_rows_and_radii(m, n, cells):
    h = 2.0 / 64
    x, y = np.meshgrid(np.arange(m) - 0.31 * m, np.arange(n) - 0.4637 * n)
    phi = (h * (np.hypot(1.01 * x, y) - 0.27 * min(m, n) - 0.013)).ravel()
    args = (m, n, -0.31 * m * h, -0.4637 * n * h, h, h, -cells * h, cells * h)
    po, so, _ = ol.build_band("oracle", *args, phi)
    pg, sg, _ = ia.build_band(*args, phi)
    assert np.array_equal(so, sg) and np.array_equal(po, pg)
