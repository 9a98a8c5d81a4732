"""Pinned host memory of the read-out: one set of slots for all contexts of a
device, given back with the last of them; a machine that has none to give still
creates runs and reads them out, with the same values.  A child process puts its
own hipHostMalloc and hipHostFree (counting, or refusing) before the library's.
Threads that read out several runs at once get each run's own state."""
import os
import shutil
import subprocess
import sys
import threading

import numpy as np
import pytest

from tests.cases import background, mhd_cfg, quiet_cfg

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SHIM = r"""
#include <stddef.h>
static int (*real_malloc)(void**, size_t, unsigned);
static int (*real_free)(void*);
static int refuse, held;
static size_t bytes;
void shim_set(void* m, void* f, int r) {
  real_malloc = (int (*)(void**, size_t, unsigned))m;
  real_free = (int (*)(void*))f;
  refuse = r;
}
size_t shim_bytes(void) { return bytes; }
int shim_held(void) { return held; }
int hipHostMalloc(void** p, size_t n, unsigned flags) {
  bytes += n;
  if (refuse) return 2;
  ++held;
  return real_malloc(p, n, flags);
}
int hipHostFree(void* p) {
  --held;
  return real_free(p);
}
"""

CHILD = r"""
import ctypes as C, re, sys
import numpy as np
shim = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
shim.shim_bytes.restype = C.c_size_t
from sparc2_amd._lib import lib
lib()
path = re.search(r"\S*libamdhip64\S*", open("/proc/self/maps").read()).group(0)
hip = C.CDLL(path)
addr = lambda f: C.cast(f, C.c_void_p)
shim.shim_set(addr(hip.hipHostMalloc), addr(hip.hipHostFree), int(sys.argv[2] == "refuse"))
from tests.cases import background, quiet_cfg, random_state
from sparc2_amd.solver import Solver
solvers, out = [], {}
for q in range(6):
    cfg = quiet_cfg(nx=64, ny=64, nz=96, precision=("fp64", "fp32")[q % 2])
    s = Solver(cfg, background(cfg))
    s.put_state(*random_state(cfg, seed=q))
    s.advance(0, 1)
    state, psi = s.get_state(with_psi=True)
    out[f"state{q}"], out[f"slab{q}"], out[f"ddx{q}"] = state, s.get_slab(1, 5, 6), s.ddx(state[0], 5)
    out[f"diag{q}"] = s.diag()
    for f, v in psi.items():
        out[f"psi{q}_{f}"] = v
    solvers.append(s)
pinned = shim.shim_bytes()
for s in solvers:
    s.close()
np.savez(sys.argv[3], **out)
print("PINNED", pinned, "HELD", shim.shim_held(), flush=True)
"""


def _child(tmp_path, mode):
    src, so = tmp_path / "shim.c", tmp_path / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", str(src), "-o", str(so)], check=True)
    result = tmp_path / f"{mode}.npz"
    r = subprocess.run([sys.executable, "-c", CHILD, str(so), mode, str(result)], cwd=ROOT, capture_output=True,
                       text=True, timeout=100)
    print(r.stdout[-2000:], r.stderr[-2000:], flush=True)
    assert r.returncode == 0
    words = r.stdout.split()
    return int(words[words.index("PINNED") + 1]), int(words[words.index("HELD") + 1]), np.load(result)


@pytest.mark.skipif(shutil.which("gcc") is None, reason="needs gcc")
def test_pinned_memory_is_shared_given_back_and_not_needed(tmp_path):
    pinned, held, with_slots = _child(tmp_path, "count")
    assert 0 < pinned <= 33 << 20  # one set of slots, and a little for each context
    assert held == 0
    refused, _, without = _child(tmp_path, "refuse")
    assert refused > 0
    assert set(with_slots.files) == set(without.files)
    for name in with_slots.files:
        np.testing.assert_array_equal(with_slots[name], without[name])


def test_threads_read_out_at_once():
    from sparc2_amd.solver import Solver
    solvers, states = [], []
    for q, (make, kw) in enumerate([(quiet_cfg, dict(nx=64, ny=64, nz=128)), (mhd_cfg, dict(nx=48, ny=40, nz=64)),
                                    (quiet_cfg, dict(nx=32, ny=32, nz=24)), (quiet_cfg, dict(nx=96, ny=64, nz=100))]):
        cfg = make(**kw)
        s = Solver(cfg, background(cfg))
        a = np.random.default_rng(q).standard_normal((cfg.nv, cfg.nz, cfg.ny, cfg.nx))
        s.put_state(a)
        solvers.append(s)
        states.append(a)
    bad = []

    def read(q):
        for k in range(5):
            if not np.array_equal(solvers[q].get_state(), states[q]):
                bad.append((q, "state"))
            if not np.array_equal(solvers[q].get_slab(2, k, k + 3), states[q][2, k:k + 4]):
                bad.append((q, "slab"))

    threads = [threading.Thread(target=read, args=(q,)) for q in range(len(solvers))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for s in solvers:
        s.close()
    assert not bad
