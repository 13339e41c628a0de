"""RR, DET and LAM asked in turn over a tau x emb grid reuse the work-item tables
of its lengths: from the second round on a call copies its series up and its
results down and nothing else.  A library loaded before the engine's counts the
copies, in a process of its own."""
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
static long copies_;
long copies(void) { return copies_; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *stream) {
    int (*f)(void *, const void *, size_t, int, void *) =
        (int (*)(void *, const void *, size_t, int, void *))dlsym(dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD),
                                                                  "hipMemcpyAsync");
    copies_++;
    return f(d, s, n, kind, stream);
}
"""

CHILD = """
import ctypes as C, sys
shim = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
shim.copies.restype = C.c_long
sys.path.insert(0, sys.argv[2])
import numpy as np, accrqa_amd as amd
for n, taus, embs in ((4001, [1, 2, 4], [2, 3, 5]), (300, [1], [2]), (2000, [1, 3], [1, 9])):
    x = np.random.default_rng(n).standard_normal(n).astype(np.float32)
    thr = np.array([0.3, 0.9], np.float32)
    for rnd in range(3):
        for f, args in ((amd.RR, ()), (amd.DET, ([2],)), (amd.LAM, ([2],))):
            before = shim.copies()
            f(x, taus, embs, *args, thr, 1)
            print(n, rnd, f.__name__, shim.copies() - before, flush=True)
"""


@pytest.mark.skipif(shutil.which("gcc") is None, reason="needs a host C compiler")
def test_grid_reuses_tables(tmp_path):
    (tmp_path / "shim.c").write_text(SHIM)
    (tmp_path / "child.py").write_text(CHILD)
    so = str(tmp_path / "shim.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", so, str(tmp_path / "shim.c"), "-ldl"], check=True)
    r = subprocess.run([sys.executable, str(tmp_path / "child.py"), so, ROOT], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
    seen = [line.split() for line in r.stdout.splitlines()]
    assert len(seen) == 27
    assert int(seen[0][3]) > 2                      # the first round builds them
    assert all(int(c) == 2 for _, rnd, _, c in seen if rnd != "0"), r.stdout
