"""The batch tuner's z chunks: for every tile shape it times the chunks the batch
takes by itself, then twice and four times them: launches of fewer and fewer
work items.  Groups whose single-run chunk differs from the batch's: small grids
(one plane alone) and rows that are not whole lines (two planes at most)."""
import ctypes as C

import pytest

from tests.cases import background, mhd_cfg, quiet_cfg

pytestmark = pytest.mark.gpu

GROUPS = {
    "mhd small": [(mhd_cfg, dict(nx=32, ny=32, nz=64)), (mhd_cfg, dict(nx=48, ny=32, nz=72))],
    "mhd odd rows": [(mhd_cfg, dict(nx=39, ny=31, nz=64)), (mhd_cfg, dict(nx=87, ny=75, nz=64))],
    "quiet": [(quiet_cfg, dict(nx=48, ny=48, nz=64)), (quiet_cfg, dict(nx=32, ny=40, nz=48))],
}


@pytest.mark.parametrize("name", GROUPS)
def test_tuner_times_deeper_and_deeper_chunks(name, monkeypatch):
    from sparc2_amd import batch
    from sparc2_amd._lib import lib
    from sparc2_amd.solver import Solver
    solvers = []
    for make, kw in GROUPS[name]:
        cfg = make(**kw)
        solvers.append(Solver(cfg, background(cfg)))
    timed = {}
    create = batch._create

    def recording(members, use_graph):
        h = create(members, use_graph)
        groups, blocks = C.c_int(), C.c_long()
        assert lib().sparc_hip_batch_info(h, C.byref(groups), C.byref(blocks)) == 0
        timed.setdefault(members[0].tile()[0][:2], []).append(blocks.value)
        return h

    monkeypatch.setattr(batch, "_create", recording)
    monkeypatch.setattr(batch, "_GROUP_CACHE", {})
    batch.tune_tiles(solvers, reps=1)
    for s in solvers:
        s.close()
    print(name, timed, flush=True)
    assert timed
    for blocks in timed.values():
        assert len(blocks) == len(batch.KC_MULT)
        assert all(a > b for a, b in zip(blocks, blocks[1:]))


@pytest.mark.parametrize("precision,cap", [("fp64", 5), ("fp32", 10)])
def test_runs_with_open_sides_keep_shallow_chunks_in_a_batch(precision, cap):
    """512 blocks of this run alone would be 21 (FP64) or 13 planes deep."""
    from sparc2_amd.solver import Solver
    cfg = quiet_cfg(nx=150, ny=150, nz=112, periodic=False, use_hpml=True, npml=(6,) * 6, precision=precision)
    s = Solver(cfg, background(cfg), tile=(32, 8, 0))
    planes = s.batch_chunk()
    s.close()
    print(precision, planes, flush=True)
    assert 2 <= planes <= cap
