"""The automatic launch geometry (tile shape, z chunk, z-pass chunk) against an
explicit one: a stage computes every point by the same arithmetic whatever the
split, so the states are equal bitwise.  Grids of one round of resident blocks,
the smallest axes among them (several rounds: test_gpu_geometry_rounds.py)."""
import numpy as np
import pytest

from tests.cases import background, mhd_cfg, quiet_cfg, random_state

pytestmark = pytest.mark.gpu

HPML = dict(periodic=False, use_hpml=True, npml=(5, 6, 6, 5, 8, 7))
CASES = {
    "quiet smallest": (quiet_cfg, dict(nx=16, ny=16, nz=17), (32, 8, 5)),
    "quiet 48": (quiet_cfg, dict(nx=48, ny=48, nz=33), (32, 8, 33)),
    "quiet 65x67 odd": (quiet_cfg, dict(nx=65, ny=67, nz=131), (64, 4, 7)),
    "quiet fp32": (quiet_cfg, dict(nx=96, ny=70, nz=64, precision="fp32"), (32, 8, 3)),
    "thermal hpml": (quiet_cfg, dict(nx=43, ny=39, nz=47, magnetic=1, **HPML), (16, 16, 47)),
    "mhd": (mhd_cfg, dict(nx=32, ny=48, nz=41), (16, 16, 7)),
    "mhd odd": (mhd_cfg, dict(nx=39, ny=31, nz=53), (32, 16, 4)),
    "mhd fp32": (mhd_cfg, dict(nx=40, ny=32, nz=40, precision="fp32"), (16, 16, 40)),
}


@pytest.mark.parametrize("name", CASES)
def test_automatic_geometry_equals_an_explicit_one(name):
    from sparc2_amd.solver import Solver
    make, kw, tile = CASES[name]
    cfg = make(**kw)
    bg = background(cfg)
    a, psi = random_state(cfg, seed=5)
    out = []
    for t in ((0, 0, 0), tile):
        s = Solver(cfg, bg, tile=t)
        print(name, t, s.tile(), flush=True)
        s.put_state(a, psi)
        s.advance(0, 6)
        out.append(s.get_state(with_psi=True))
        s.close()
    assert np.array_equal(out[0][0], out[1][0])
    for f in out[0][1]:
        assert np.array_equal(out[0][1][f], out[1][1][f])
