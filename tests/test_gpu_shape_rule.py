"""The automatic tile of quiet runs whose rows are not whole 128-byte lines: grids
where a shape was measured 15 to 60 % slower than another one (a step in us, by
shape: FP32 79x134x136 16x16 297, 32x8 229; 69x229x144 16x16 491, 64x4 379;
89x267x239 32x8 811, 32x16 673; FP64 110x125x186 16x16 540, 32x16 464) do not get
that shape."""
import pytest

from tests.cases import background, quiet_cfg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size,precision,slow", [((79, 134, 136), "fp32", (16, 16)), ((69, 229, 144), "fp32", (16, 16)),
                                                 ((89, 267, 239), "fp32", (32, 8)), ((110, 125, 186), "fp64", (16, 16))])
def test_slow_shape_is_not_taken(size, precision, slow):
    from sparc2_amd.solver import Solver
    nx, ny, nz = size
    cfg = quiet_cfg(nx=nx, ny=ny, nz=nz, precision=precision)
    s = Solver(cfg, background(cfg))
    tile, blocks = s.tile()
    s.close()
    print(size, precision, tile, blocks, flush=True)
    assert tile[:2] != slow
