"""FFT damping of planes that a block transforms in LDS, against the oracle's
direct DFT sums: radices at the ends and inside of a transform (radix 2 is in
test_gpu_damping_paths.py), odd sides, one to three passes, padded and unpadded
slabs, and both block sizes.  Bars as in test_gpu_damping.py: FP64
relative L2 1e-11 per field after the steps, FP32 within 1e-5 of FP64."""
import numpy as np
import pytest

from oracle.oracle import Oracle
from tests.cases import background, field_errors, quiet_cfg, random_state

pytestmark = pytest.mark.gpu

SIZES = [(32, 24, 16), (24, 50, 17), (36, 28, 16), (49, 45, 16), (27, 40, 19), (144, 16, 16),
         (20, 112, 16), (42, 18, 21), (60, 42, 16), (128, 90, 16)]


def _run(cfg, bg, a, psi):
    from sparc2_amd.solver import Solver
    s = Solver(cfg, bg)
    s.put_state(a, psi)
    s.advance(0, 3)
    out = s.get_state()
    s.close()
    return out


@pytest.mark.parametrize("nx,ny,nz", SIZES)
def test_planes_in_lds_match_oracle(nx, ny, nz):
    cfg = quiet_cfg(nx=nx, ny=ny, nz=nz, damping=True)
    bg = background(cfg)
    a, psi = random_state(cfg, seed=29)
    o = Oracle(cfg, bg)
    o.put_state(a)
    for f, v in psi.items():
        o.put_psi(f, v)
    o.run(0, 3)
    print(nx, ny, nz, flush=True)
    ref = o.get_state()
    got = _run(cfg, bg, a, psi)
    assert max(field_errors(got, ref)) < 1e-11
    single = _run(cfg.replace(precision="fp32"), bg, a, psi)
    assert max(field_errors(single, got)) < 1e-5
    assert not np.array_equal(single, got)
