"""FILTER_VARS where a wave's ring of rows turns: enough planes that a wave of the
fused y and x filter marches 32 or 64 rows (the ring holds 17 rows with 11 points,
13 with 7; small grids march 16), and grids of odd nx * ny, whose FP32 z filter
takes one column a lane.  Bars as in test_gpu_filters.py: FP64 against the oracle
1e-13, FP32 within 1e-6 of FP64."""
import pytest

from oracle.oracle import Oracle
from tests.cases import background, field_errors, mhd_cfg, quiet_cfg, random_state

pytestmark = pytest.mark.gpu

G3 = dict(filter_mode_xy=2, filter_mode_z=2, s_xy=0.7, s_z=0.6)
HPML = dict(periodic=False, use_hpml=True, npml=(6, 6, 6, 6, 8, 8))

CASES = {
    "11 points, 32 rows, periodic": lambda: quiet_cfg(nx=70, ny=70, nz=280),
    "11 points, 64 rows, periodic": lambda: quiet_cfg(nx=53, ny=71, nz=420),
    "11 points, 32 rows, odd, open": lambda: quiet_cfg(nx=55, ny=87, nz=280, **HPML),
    "7 points, 64 rows, odd, open": lambda: mhd_cfg(nx=57, ny=71, nz=264, **G3),
    "7 points, 32 rows, odd, periodic": lambda: quiet_cfg(nx=59, ny=67, nz=280, **G3),
}


@pytest.mark.parametrize("case", CASES)
def test_filters_over_turns_of_the_ring(case):
    from sparc2_amd.solver import Solver
    cfg = CASES[case]()
    bg = background(cfg)
    a, _ = random_state(cfg, seed=19)
    t = cfg.xyfreq * cfg.zfreq
    o = Oracle(cfg, bg)
    o.put_state(a)
    o.filter_vars(t)
    ref = o.get_state()
    s = Solver(cfg, bg)
    s.put_state(a)
    s.filter_vars(t)
    got = s.get_state()
    errs = field_errors(got, ref)
    s32 = Solver(cfg.replace(precision="fp32"), bg, setup=s.st)
    s32.put_state(a)
    s32.filter_vars(t)
    e32 = field_errors(s32.get_state(), got)
    print(case, "FP64 " + " ".join(f"{e:.1e}" for e in errs), "FP32 " + " ".join(f"{e:.1e}" for e in e32), flush=True)
    s32.close()
    s.close()
    assert max(errs) < 1e-13
    assert max(e32) < 1e-6
