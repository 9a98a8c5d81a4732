"""A batch whose runs are cut into more blocks behind its back, by set_tile and by
a second batch (their buffers of diagnostic partials are replaced by longer ones):
states, diagnostics and the failure record stay those of a batch left alone."""
import numpy as np
import pytest

from tests.cases import background, mhd_cfg, random_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("use_graph", [False, True])
def test_batch_survives_longer_partials_of_its_runs(use_graph):
    from sparc2_amd.batch import Batch
    from sparc2_amd.solver import Solver
    sets = []
    for _ in range(2):
        solvers = []
        for q, n in enumerate([(32, 48, 56), (39, 31, 53)]):
            cfg = mhd_cfg(nx=n[0], ny=n[1], nz=n[2])
            s = Solver(cfg, background(cfg), tile=(16, 16, 8))
            s.put_state(*random_state(cfg, seed=50 + q))
            solvers.append(s)
        sets.append((solvers, Batch(solvers, use_graph=use_graph)))
    (kept, alone), (moved, batch) = sets
    for b in (alone, batch):
        b.advance(2)
    for s in moved:
        before = s.tile()[1]
        s.set_tile((16, 16, 1))
        assert s.tile()[1] > before
    second = Batch(moved[:1], use_graph=False)
    for b in (alone, batch):
        assert b.advance(3) == {}
    second.close()
    for one, other in zip(kept, moved):
        np.testing.assert_array_equal(one.get_state(), other.get_state())
        np.testing.assert_array_equal(one.diag(), other.diag())
        assert one.guard()[0] == other.guard()[0]
    for solvers, b in sets:
        b.close()
        for s in solvers:
            s.close()
