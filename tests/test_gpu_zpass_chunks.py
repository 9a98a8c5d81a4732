"""The z pass of an MHD stage cut into chunks of equal work: a run alone and
the same run in a batch, whose chunks are fewer and deeper, agree bitwise.
Layer widths from none to nearly the whole axis, an axis of few planes, and
columns that do not fill their blocks."""
import numpy as np
import pytest

from tests.cases import background, mhd_cfg, random_state

pytestmark = pytest.mark.gpu

SIZES = [  # nx, ny, nz, z layer widths (bottom, top)
    (24, 22, 29, (10, 10)), (39, 31, 97, (10, 10)), (32, 24, 40, (0, 12)),
    (24, 40, 53, (25, 26)), (40, 23, 121, (3, 0)), (32, 32, 64, (0, 0)),
]


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("nx,ny,nz,layers", SIZES)
def test_chunks_of_the_z_pass_do_not_change_the_state(nx, ny, nz, layers, precision):
    from sparc2_amd.batch import Batch
    from sparc2_amd.solver import Solver
    cfg = mhd_cfg(nx=nx, ny=ny, nz=nz, precision=precision, periodic=False, use_hpml=True,
                  npml=(5, 5, 6, 6) + layers)
    bg = background(cfg)
    a, psi = random_state(cfg, seed=9)
    alone, member = Solver(cfg, bg), Solver(cfg, bg)
    print(nx, ny, nz, layers, precision, alone.tile(), flush=True)
    alone.put_state(a, psi)
    member.put_state(a, psi)
    batch = Batch([member])
    alone.advance(0, 4)
    batch.advance(5)
    x, px = alone.get_state(with_psi=True)
    y, py = member.get_state(with_psi=True)
    batch.close()
    assert np.array_equal(x, y)
    for f in px:
        assert np.array_equal(px[f], py[f])
