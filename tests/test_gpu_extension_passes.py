"""The extension ends in about one launch however its tiles depend on each
other: the tiles of a lattice of blobs and of bands many tiles deep, more of them
than workgroups, also where fits' windows grow (spacings of a few 1e-6), bit for
bit against the oracle's serial extrapolate_fields.
Every tile is held by a workgroup that runs, so one launch is enough; the
bound leaves room for a workgroup that gave up early. (Sweeps over all tiles
take a launch for each tile boundary on the longest chain: 16 to about 150 here.)"""
import numpy as np
import pytest

from tests.test_gpu_extension import _compare, wavy

pytestmark = pytest.mark.gpu


def _tiles(s, m, n):
    j, i = np.nonzero((s.reshape(n, m) == 4) | (s.reshape(n, m) == 5))
    return np.unique(j // 16 * m + i // 16).size


def _star(r, a):
    return lambda x, y: np.hypot(x, y) - r - a * np.sin(5 * np.arctan2(y, x) + 0.4)


def _blobs(x, y):
    return 50 / np.pi * (0.35 + 0.03 * np.sin(0.013 * x + 0.02 * y) - np.cos(np.pi * x / 50) * np.cos(np.pi * y / 50))


@pytest.mark.parametrize("m,n,h,shape,cells,tiles", [
    (63, 50, 2.5e-3, wavy, 7.0, 1), (803, 811, 2.5e-3, _blobs, 6.0, 1500), (700, 700, 2.5e-3, _star(200, 30), 100.0, 769),
    (1200, 1180, 2.5e-3, _star(340, 50), 160.0, 1900), (250, 260, 8e-6, _star(70, 12), 7.0, 40),
    (700, 690, 4e-6, _star(200, 30), 40.0, 300), (803, 811, 8e-6, _blobs, 5.0, 1500),
    (1400, 1400, 8e-6, _star(400, 60), 60.0, 769)])
def test_about_one_launch(m, n, h, shape, cells, tiles):
    s, passes = _compare(m, n, h, shape, cells)
    assert _tiles(s, m, n) >= tiles
    assert passes <= 4
