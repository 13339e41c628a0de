"""DET asked alone where the rank-tile store's memory cannot be had: the call
takes the form without a store and returns that form's results.  A library
loaded before the engine's takes hipMalloc over and turns requests above a limit
into one the runtime refuses, in a process of its own."""
import os
import shutil
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SHIM = """
#include <dlfcn.h>
#include <stddef.h>
static size_t limit_ = (size_t)-1, refused_;
void limit(size_t b) { limit_ = b; }
size_t refused(void) { return refused_; }
int hipMalloc(void **p, size_t n) {
    int (*f)(void **, size_t) = (int (*)(void **, size_t))dlsym(dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD), "hipMalloc");
    if (n > limit_) refused_++;
    return f(p, n > limit_ ? (size_t)1 << 48 : n);
}
"""

CHILD = """
import ctypes as C, sys
shim = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
shim.limit.argtypes, shim.refused.restype = [C.c_size_t], C.c_size_t
sys.path.insert(0, sys.argv[2])
import numpy as np, accrqa_amd as amd
m = 16
# a larger store for the second type; N_c^2 / 2 bytes
for dt, nc in ((np.float32, 20000), (np.float64, 30000)):
    w = np.cumsum(np.random.default_rng(nc).standard_normal(nc + m - 1))
    x, thr = ((w - w.mean()) / w.std()).astype(dt), np.array([1.5, 3.0], dt)
    amd.set_split(amd.SPLIT_NEVER)
    want = amd.DET(x, [1], [m], [2], thr, 1)
    amd.set_split(amd.SPLIT_AUTO)
    shim.limit(nc * nc // 4)
    before = shim.refused()
    got = amd.DET(x, [1], [m], [2], thr, 1)
    assert shim.refused() == before + 1, "the store was not asked for"
    assert amd.load().accrqa_amd_last_error() == b""
    shim.limit(C.c_size_t(-1).value)
    again = amd.DET(x, [1], [m], [2], thr, 1)
    assert np.array_equal(got, want) and np.array_equal(again, want), (dt, got, again, want)
    print("same", dt.__name__, flush=True)
"""


@pytest.mark.skipif(shutil.which("gcc") is None, reason="needs a host C compiler")
def test_det_alone_without_the_store(tmp_path):
    (tmp_path / "shim.c").write_text(SHIM)
    (tmp_path / "child.py").write_text(CHILD)
    so = str(tmp_path / "shim.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", so, str(tmp_path / "shim.c"), "-ldl"], check=True)
    r = subprocess.run([sys.executable, str(tmp_path / "child.py"), so, ROOT], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.split() == ["same", "float32", "same", "float64"]
