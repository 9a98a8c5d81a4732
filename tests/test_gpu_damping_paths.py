"""FFT damping on both paths of the dispatch, in both precisions, against the
oracle's direct DFT sums: the library's transforms for sides with a prime factor
above 7 (three fields in one plan on unpadded slabs, one on padded ones) and for
planes that LDS does not hold; planes of 150 to 158 of its 160 KB; sides of 98,
the one size up to 400 with a pass of radix 2, along x and along y.  Bars as in
test_gpu_damping.py: FP64 relative L2 1e-11 per field, FP32 within 1e-5 of FP64.
The box grows with the grid: the damping's rate grows with the wavenumber, and
cells much smaller than these take its rate times the time step out of the
scheme's stable range, where a step amplifies rounding."""
import numpy as np
import pytest

from oracle.oracle import Oracle
from tests.cases import background, field_errors, quiet_cfg, random_state

pytestmark = pytest.mark.gpu

SIZES = [(33, 32, 25),    # library, padded
         (32, 33, 24),    # library, unpadded
         (160, 160, 16),  # FP64: too large for LDS; FP32: 106 KB
         (200, 200, 16),  # too large in both
         (144, 128, 16),  # FP64: 152 KB
         (160, 120, 16),  # FP64: 158 KB
         (192, 200, 16),  # FP32: 156 KB
         (98, 40, 16), (40, 98, 17)]


def _run(cfg, bg, a, psi):
    from sparc2_amd.solver import Solver
    s = Solver(cfg, bg)
    s.put_state(a, psi)
    s.advance(0, 1)
    out = s.get_state()
    s.close()
    return out


@pytest.mark.parametrize("nx,ny,nz", SIZES)
def test_damping_paths_match_oracle(nx, ny, nz):
    cfg = quiet_cfg(nx=nx, ny=ny, nz=nz, damping=True, xlength=25e8 * nx / 48, ylength=25e8 * ny / 48)
    bg = background(cfg)
    a, psi = random_state(cfg, seed=31)
    o = Oracle(cfg, bg)
    o.put_state(a)
    for f, v in psi.items():
        o.put_psi(f, v)
    o.run(0, 1)
    print(nx, ny, nz, flush=True)
    ref = o.get_state()
    got = _run(cfg, bg, a, psi)
    errs = field_errors(got, ref)
    single = _run(cfg.replace(precision="fp32"), bg, a, psi)
    errs32 = field_errors(single, got)
    print("FP64 " + " ".join(f"{e:.1e}" for e in errs) + "  FP32 " + " ".join(f"{e:.1e}" for e in errs32), flush=True)
    assert max(errs) < 1e-11
    assert max(errs32) < 1e-5
    assert not np.array_equal(single, got)
