"""The automatic launch geometry on grids of more than one round of resident
blocks, where the caps on the z chunk bind: open sides (at most 5 planes in FP64),
the MHD xy kernel with rows of whole lines (at most 6, FP32 5) and without (at
most 2), and deep quiet chunks.  As in test_gpu_geometry.py the states are bitwise
those of an explicit geometry."""
import numpy as np
import pytest

from tests.cases import background, mhd_cfg, quiet_cfg, random_state

pytestmark = pytest.mark.gpu

HPML = dict(periodic=False, use_hpml=True, npml=(5, 6, 6, 5, 8, 7))
# run, explicit tile, planes a chunk may have, whether two rounds are meant
CASES = {
    "quiet deep": (quiet_cfg, dict(nx=192, ny=160, nz=96), (16, 16, 11), (2, 96), False),
    "quiet two rounds": (quiet_cfg, dict(nx=300, ny=260, nz=40), (32, 8, 7), (2, 40), True),
    "thermal open": (quiet_cfg, dict(nx=150, ny=118, nz=64, magnetic=1, **HPML), (32, 16, 64), (2, 5), True),
    "thermal open fp32": (quiet_cfg, dict(nx=190, ny=150, nz=64, magnetic=1, precision="fp32", **HPML),
                          (16, 16, 3), (2, 10), False),
    "mhd lines": (mhd_cfg, dict(nx=128, ny=112, nz=100), (32, 8, 9), (2, 6), True),
    "mhd other rows": (mhd_cfg, dict(nx=121, ny=118, nz=64), (16, 16, 5), (2, 2), True),
    "mhd lines fp32": (mhd_cfg, dict(nx=160, ny=150, nz=80, precision="fp32"), (16, 16, 13), (2, 5), True),
}


@pytest.mark.parametrize("name", CASES)
def test_geometry_of_several_rounds_equals_an_explicit_one(name):
    from sparc2_amd.solver import Solver
    make, kw, tile, (least, most), rounds = CASES[name]
    cfg = make(**kw)
    bg = background(cfg)
    a, psi = random_state(cfg, seed=7)
    out, tiles = [], []
    for t in ((0, 0, 0), tile):
        s = Solver(cfg, bg, tile=t)
        tiles.append(s.tile())
        s.put_state(a, psi)
        s.advance(0, 2)
        out.append(s.get_state(with_psi=True))
        s.close()
    print(name, tiles, flush=True)
    (shape, blocks), (explicit, _) = tiles
    assert shape != explicit and explicit == tile
    assert least <= shape[2] <= most
    # at most 512 blocks of these tiles are resident at once
    assert (blocks > 512) == rounds
    assert np.array_equal(out[0][0], out[1][0])
    for f in out[0][1]:
        assert np.array_equal(out[0][1][f], out[1][1][f])
