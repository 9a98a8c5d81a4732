"""FFT damping where the field slabs are padded and where they are not (where the
library transforms the planes: each field by itself, or three in one), against
the oracle's direct DFT sums; odd and even plane sizes.  Bar as in
test_gpu_damping.py: FP64 relative L2 1e-11 per field after the steps."""
import pytest

from oracle.oracle import Oracle
from tests.cases import background, field_errors, quiet_cfg, random_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz", [(33, 32, 25), (32, 33, 24), (17, 19, 21), (16, 16, 16)])
def test_damped_planes_match_oracle(nx, ny, nz):
    from sparc2_amd.solver import Solver
    cfg = quiet_cfg(nx=nx, ny=ny, nz=nz, damping=True)
    bg = background(cfg)
    a, psi = random_state(cfg, seed=23)
    o = Oracle(cfg, bg)
    o.put_state(a)
    for f, v in psi.items():
        o.put_psi(f, v)
    o.run(0, 5)
    print(nx, ny, nz, "padded" if nx * ny * nz % 256 else "unpadded", flush=True)
    s = Solver(cfg, bg)
    s.put_state(a, psi)
    s.advance(0, 5)
    errs = field_errors(s.get_state(), o.get_state())
    s.close()
    assert max(errs) < 1e-11
