"""Device memory refused where a run is cut into more blocks (set_tile, or a
batch): the call fails, and the run keeps its geometry and goes on as before.  A
child process puts its own hipMalloc before the library's."""
import os
import shutil
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SHIM = r"""
#include <stddef.h>
static int (*real_malloc)(void**, size_t);
static size_t limit;
void shim_set(void* m, size_t n) {
  real_malloc = (int (*)(void**, size_t))m;
  limit = n;
}
int hipMalloc(void** p, size_t n) { return limit && n == limit ? 2 : real_malloc(p, n); }
"""

CHILD = r"""
import ctypes as C, re, sys
import numpy as np
shim = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
from sparc2_amd._lib import SparcError, lib
lib()
hip = C.CDLL(re.search(r"\S*libamdhip64\S*", open("/proc/self/maps").read()).group(0))
refuse = lambda n: shim.shim_set(C.cast(hip.hipMalloc, C.c_void_p), C.c_size_t(n))
refuse(0)
from sparc2_amd.batch import Batch
from sparc2_amd.solver import Solver
from tests.cases import background, mhd_cfg, random_state

def made():
    cfg = mhd_cfg(nx=96, ny=64, nz=96)
    s = Solver(cfg, background(cfg))
    s.put_state(*random_state(cfg, seed=3))
    return s

def refused(call, blocks):
    refuse(24 * blocks)
    try:
        call()
    except SparcError as e:
        print("refused:", e, flush=True)
    else:
        raise SystemExit("not refused")
    refuse(0)

one, other = made(), made()
before = one.tile()
# one plane a chunk: 6 x 4 tiles of 16 x 16, 96 planes
assert before[1] < 6 * 4 * 96
refused(lambda: one.set_tile((16, 16, 1)), 6 * 4 * 96)
assert one.tile() == before
one.advance(0, 1)
other.advance(0, 1)
assert np.array_equal(one.get_state(), other.get_state())
# a batch cuts it by its own rule
chunk = one.batch_chunk()
blocks = 6 * 4 * -(-96 // chunk)
print("alone", before, "batch", chunk, blocks, flush=True)
assert blocks > before[1]
refused(lambda: Batch([one]), blocks)
assert one.tile() == before
one.advance(2, 3)
other.advance(2, 3)
assert np.array_equal(one.get_state(), other.get_state())
one.close()
other.close()
print("WELL", flush=True)
"""


@pytest.mark.skipif(shutil.which("gcc") is None, reason="needs gcc")
def test_a_refused_cut_leaves_the_run_as_it_was(tmp_path):
    src, so = tmp_path / "shim.c", tmp_path / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", str(src), "-o", str(so)], check=True)
    r = subprocess.run([sys.executable, "-c", CHILD, str(so)], cwd=ROOT, capture_output=True, text=True, timeout=100)
    print(r.stdout[-2000:], r.stderr[-2000:], flush=True)
    assert r.returncode == 0 and "WELL" in r.stdout
