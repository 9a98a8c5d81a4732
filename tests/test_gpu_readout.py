"""Read-out of the state: what put_state stored comes back exactly, over array
sizes around the pieces the copies are cut into (one short piece, ragged last
pieces, several workers).  FP32: the compensated value a - c in FP64, with
a = fl32(x) and c = bf16(fl32(a - x)) (bfloat16, nearest even)."""
import numpy as np
import pytest

from tests.cases import background, mhd_cfg, quiet_cfg

pytestmark = pytest.mark.gpu


def _bf16(x):
    u = x.astype(np.float32).view(np.uint32)
    u = u + (0x7FFF + ((u >> 16) & 1)).astype(np.uint32)
    return (u & np.uint32(0xFFFF0000)).view(np.float32)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("make,size", [(quiet_cfg, (16, 16, 16)), (mhd_cfg, (31, 40, 37)),
                                       (quiet_cfg, (64, 64, 128)), (mhd_cfg, (96, 80, 131))])
def test_state_comes_back(make, size, precision):
    from sparc2_amd.solver import Solver
    nx, ny, nz = size
    cfg = make(nx=nx, ny=ny, nz=nz, precision=precision)
    s = Solver(cfg, background(cfg))
    rng = np.random.default_rng(3)
    a = rng.standard_normal((cfg.nv, nz, ny, nx)) * 10.0 ** rng.integers(-6, 3, (cfg.nv, 1, 1, 1))
    psi = {f: rng.standard_normal(s.face_shape(f)) for f in range(6) if cfg.face_active(f)}
    s.put_state(a, psi)
    print(size, precision, flush=True)
    got, gpsi = s.get_state(with_psi=True)
    if precision == "fp64":
        want, wpsi = a, psi
    else:
        hi = a.astype(np.float32)
        want = hi.astype(np.float64) - _bf16((hi.astype(np.float64) - a).astype(np.float32)).astype(np.float64)
        wpsi = {f: v.astype(np.float32).astype(np.float64) for f, v in psi.items()}
    assert np.array_equal(got, want)
    for f, v in wpsi.items():
        assert np.array_equal(gpsi[f], v)
    # planes of one field, from an offset that is no multiple of a piece
    assert np.array_equal(s.get_slab(cfg.nv - 1, 3, nz - 2), want[cfg.nv - 1, 3:nz - 1])
    s.close()
