"""The one-launch extension (every point evaluated once, when what it reads is
final) against the oracle's serial extrapolate_fields, bit for bit, where the
kernel takes another route than in the ordinary shapes: remainders of tiles,
fits whose window grows past radius 3, more active tiles than workgroups, and
a fit that stays singular."""
import numpy as np
import pytest

import incrmt_amd as ia
from tests import oracle_lib as ol

pytestmark = pytest.mark.gpu


def _case(m, n, h, phi_of, cells=7.0):
    x, y = np.meshgrid(np.arange(m) - 0.47 * m, np.arange(n) - 0.53 * n)
    phi = h * phi_of(x, y)
    args = (m, n, -0.47 * m * h, -0.53 * n * h, h, h, -cells * h, cells * h)
    fx = np.where(phi < 0, 1 + 0.3 * x - 0.01 * x * y, 0.0)
    fy = np.where(phi < 0, np.sin(0.2 * x) + 0.1 * y, 0.0)
    return args, phi.ravel(), fx.ravel(), fy.ravel()


def _compare(m, n, h, phi_of, cells=7.0):
    args, phi, fx, fy = _case(m, n, h, phi_of, cells)
    rc, po, so, ex, ey = ol.build_band_extrapolate("oracle", *args, phi, fx, fy)
    assert rc == 0
    pg, sg, gx, gy, passes = ia.extrapolate(*args, phi, fx, fy)
    assert np.array_equal(so, sg) and np.array_equal(po, pg)
    assert np.array_equal(ex, gx) and np.array_equal(ey, gy)
    return sg, passes


def wavy(x, y):
    return np.hypot(x, y) - 14.3 - 2.1 * np.sin(5 * np.arctan2(y, x) + 0.4)


@pytest.mark.parametrize("m,n", [(48, 48), (49, 47), (63, 50), (65, 64), (80, 81), (47, 97)])
def test_tile_remainders(m, n):
    _compare(m, n, 2.0 / 64, wavy)


# the fit's determinant is compared with 1e-10 whatever the grid's spacing:
# at these spacings part of the windows, or all of them, grow
@pytest.mark.parametrize("h", [3e-5, 8e-6, 4e-6, 2e-6])
def test_windows_grow(h):
    _compare(61, 66, h, wavy)


def test_singular_fit_is_reported():
    args, phi, fx, fy = _case(61, 66, 1e-8, wavy)
    rc = ol.build_band_extrapolate("oracle", *args, phi, fx, fy)[0]
    assert rc != 0
    with pytest.raises(ia.IncrmtError) as e:
        ia.extrapolate(*args, phi, fx, fy)
    assert e.value.code == ia.ERR_SINGULAR_FIT


def test_more_tiles_than_workgroups():
    """A lattice of 16 x 16 blobs: about 1700 of the tiles hold points of the
    outside band, so workgroups go through several tiles each."""
    def blobs(x, y):
        u, v = x / 50.0, y / 50.0
        return 50 / np.pi * (0.35 + 0.03 * np.sin(0.013 * x + 0.02 * y) - np.cos(np.pi * u) * np.cos(np.pi * v))
    s, passes = _compare(803, 811, 2.0 / 800, blobs, cells=6.0)
    tiles = np.zeros((51, 51), bool)
    j, i = np.nonzero((s.reshape(811, 803) == 4) | (s.reshape(811, 803) == 5))
    tiles[j // 16, i // 16] = True
    assert tiles.sum() > 1024
    assert passes < 200
