"""FFT damping through the library where device memory for the three fields'
spectra together is refused (a child process puts its own hipMalloc before the
library's): the fields are then transformed one by one, as they are where the
slabs are padded.  Bar as in test_gpu_damping.py: FP64 relative L2 1e-11 per field
against the oracle."""
import os
import shutil
import subprocess
import sys

import numpy as np
import pytest

from oracle.oracle import Oracle
from tests.cases import background, field_errors, quiet_cfg, random_state

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
NX, NY, NZ = 32, 33, 24  # 33 = 3 * 11: the library's path; unpadded slabs

SHIM = r"""
#include <stddef.h>
static int (*real_malloc)(void**, size_t);
static size_t limit;
static int refused;
void shim_set(void* m, size_t n) {
  real_malloc = (int (*)(void**, size_t))m;
  limit = n;
}
int shim_refused(void) { return refused; }
int hipMalloc(void** p, size_t n) {
  if (limit && n == limit) {
    ++refused;
    return 2;
  }
  return real_malloc(p, n);
}
"""

CHILD = r"""
import ctypes as C, re, sys
import numpy as np
shim = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
from sparc2_amd._lib import lib
lib()
hip = C.CDLL(re.search(r"\S*libamdhip64\S*", open("/proc/self/maps").read()).group(0))
shim.shim_set(C.cast(hip.hipMalloc, C.c_void_p), C.c_size_t(int(sys.argv[2])))
from tests.cases import background, quiet_cfg, random_state
from sparc2_amd.solver import Solver
cfg = quiet_cfg(nx=%d, ny=%d, nz=%d, damping=True)
s = Solver(cfg, background(cfg))
s.put_state(*random_state(cfg, seed=23))
s.advance(0, 5)
np.save(sys.argv[3], s.get_state())
s.close()
print("REFUSED", shim.shim_refused(), flush=True)
""" % (NX, NY, NZ)


@pytest.mark.skipif(shutil.which("gcc") is None, reason="needs gcc")
def test_damping_one_field_at_a_time_where_memory_is_short(tmp_path):
    src, so, out = tmp_path / "shim.c", tmp_path / "shim.so", tmp_path / "state.npy"
    src.write_text(SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", str(src), "-o", str(so)], check=True)
    spectra = 3 * NZ * NY * (NX // 2 + 1) * 16
    r = subprocess.run([sys.executable, "-c", CHILD, str(so), str(spectra), str(out)], cwd=ROOT, capture_output=True,
                       text=True, timeout=100)
    print(r.stdout[-1000:], r.stderr[-2000:], flush=True)
    assert r.returncode == 0
    assert "REFUSED 1" in r.stdout
    cfg = quiet_cfg(nx=NX, ny=NY, nz=NZ, damping=True)
    a, psi = random_state(cfg, seed=23)
    o = Oracle(cfg, background(cfg))
    o.put_state(a)
    for f, v in psi.items():
        o.put_psi(f, v)
    o.run(0, 5)
    assert max(field_errors(np.load(out), o.get_state())) < 1e-11
