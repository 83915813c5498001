"""The tile of the level-set passes is a build parameter (INCRMT_LS_TILE_X and
_Y): any whole number of wavefronts up to 1024 threads, at least 8 rows. The
extension takes a tile in parts where a row of it does not fit its flags, or
its wavefronts and one more not a workgroup."""
import os
import subprocess

import pytest

from incrmt_amd import build

try:
    HIPCC = build.hipcc()
except RuntimeError:
    HIPCC = None


@pytest.mark.skipif(HIPCC is None, reason="no hipcc")
@pytest.mark.parametrize("x,y", [(8, 8), (4, 16), (26, 32), (28, 16), (30, 32), (32, 8), (128, 8), (64, 16), (16, 64)])
def test_builds(tmp_path, x, y):
    src = tmp_path / "threads.hip"
    src.write_text(f'#include "{os.path.join(build.CSRC, "levelset.hip")}"\n'
                   'namespace incrmt { namespace {\n'
                   'static_assert(kExtThreads <= 1024 && kEW <= 32, "");\n'
                   'static_assert(kExtPerTile * (kExtThreads - 64) == kTileThreads, "");\n}}\n')
    r = subprocess.run([HIPCC, f"--offload-arch={build.ARCH}", "-std=c++17", "-w", "-fsyntax-only",
                        f"-DINCRMT_LS_TILE_X={x}", f"-DINCRMT_LS_TILE_Y={y}", str(src)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
