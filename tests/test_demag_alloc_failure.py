"""Demag plans on a stand-in runtime, loaded in front of the real one in a child
process: it hands out fake addresses, fails chosen allocations and counts
calls; nothing reaches a GPU.

- A device allocation that fails during plan creation is reported, and no kernel
  is launched with a missing table.
- Reading the octant of a plan makes no pinned buffers for less than 48 MB."""
import os
import subprocess
import sys

import pytest

from hotspin_amd import _lib

SHIM = r"""
#include <stdlib.h>
#include <string.h>
static long pinned;
long shim_pinned(void) { return pinned; }
int hipHostMalloc(void** p, size_t n, unsigned f) { pinned++; *p = malloc(n); return 0; }
int hipHostFree(void* p) { free(p); return 0; }
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipSetDevice(int d) { return 0; }
int hipPointerGetAttributes(void* a, const void* p) { return 1; }
int hipEventCreateWithFlags(void** e, unsigned f) { *e = e; return 0; }
int hipEventDestroy(void* e) { return 0; }
int hipEventRecord(void* e, void* st) { return 0; }
int hipEventSynchronize(void* e) { return 0; }
static long calls, fail_from = -1, fail_to, live, launches_after, failed;
void shim_fail(long from, long to) { calls = launches_after = failed = 0; fail_from = from; fail_to = to; }
long shim_calls(void) { return calls; }
long shim_live(void) { return live; }
long shim_launches_after_failure(void) { return launches_after; }
int hipMalloc(void** p, size_t n) {
    long k = calls++;
    if (k >= fail_from && k < fail_to) { failed = 1; return 2; }
    *p = malloc(1); live++; return 0;
}
int hipFree(void* p) { if (p) { free(p); live--; } return 0; }
int hipMemcpy(void* d, const void* s, size_t n, int kind) { return 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void* st) { if (kind == 2) memset(d, 0, n); return 0; }
int hipMemsetAsync(void* d, int v, size_t n, void* st) { return 0; }
int hipStreamSynchronize(void* st) { return 0; }
int hipGetLastError(void) { return 0; }
int hipFuncSetAttribute(const void* f, int a, int v) { return 0; }
int hipLaunchKernel(const void* f, unsigned long long g, unsigned gz, unsigned long long b, unsigned bz, void** a,
                    size_t s, void* st) { launches_after += failed; return 0; }
"""

LOAD = """
import ctypes as C, sys
sys.path.insert(0, {root!r})
shim = C.CDLL({shim!r}, C.RTLD_GLOBAL)
for f in (shim.shim_calls, shim.shim_live, shim.shim_launches_after_failure, shim.shim_pinned):
    f.restype = C.c_long
shim.shim_fail.argtypes = [C.c_long, C.c_long]
from hotspin_amd import _lib
L = _lib.lib()
"""

FAILURES = LOAD + """
def plan(N, lo, hi):
    shim.shim_fail(lo, hi)
    d = L.hs_demag_create((C.c_int * 3)(*N), (C.c_double * 3)(2e-9, 2e-9, 2e-9), (C.c_int * 3)(0, 0, 0), 6, None)
    out = d, L.hs_last_error(), shim.shim_calls(), shim.shim_launches_after_failure()
    L.hs_clear_error()
    if d:
        L.hs_demag_destroy(d)
    assert shim.shim_live() == 0, (N, lo, "device memory left behind")
    return out
for N in {meshes!r}:
    d, err, n, _ = plan(N, -1, -1)
    # each allocation of some MB costs up to 0.2 ms: tables, octants, spectra and one for all temporaries
    assert d and not err and 5 <= n <= 8, (N, err, n)
    for k in range(n):  # from allocation k on: the retry of a padded plan at its logic size fails too
        d, err, _, launches = plan(N, k, 1 << 30)
        assert not d and err == 10004 and launches == 0, (N, k, err, launches)
    if {single!r}:
        for k in range(n):  # allocation k alone, where there is no retry
            d, err, _, launches = plan(N, k, k + 1)
            assert not d and err == 10004 and launches == 0, (N, k, err, launches)
    else:
        for k in range(n):  # ... and where the retry gets what it asks for
            d, err, calls, _ = plan(N, k, k + 1)
            assert d and not err and calls > n, (N, k, err, calls)
print("fine")
"""


def _no_gpu():
    try:
        import torch
        return not torch.cuda.is_available()
    except Exception:
        return True


OCTANT = LOAD + """
from hotspin_amd.api import Demag
for N, pinned in {meshes!r}:
    d = Demag(N, (2e-9,) * 3)
    before = shim.shim_pinned()
    d.kernel()
    assert shim.shim_pinned() - before == pinned, (N, shim.shim_pinned() - before)
    d.close()
print("fine")
"""

pytestmark = pytest.mark.skipif(not os.path.exists(_lib.LIB_PATH) or not _no_gpu(),
                                reason="host-side check: needs the built library and no GPU")


def _run(tmp_path, child, **values):
    src, so = tmp_path / "shim.c", tmp_path / "shim.so"
    src.write_text(SHIM)
    subprocess.check_call(["gcc", "-shared", "-fPIC", "-O1", "-w", "-o", str(so), str(src)])
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", child.format(root=root, shim=str(so), **values)], capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.strip() == "fine", r.stdout + r.stderr


# three kernels; padded lengths in three kernels and in five passes; run-time lengths
# (a one-cell axis).  None of these plans times its passes, which takes real events.
@pytest.mark.parametrize("meshes,single", [([(2, 8, 16), (4, 64, 64)], True), ([(7, 75, 100), (3, 9, 7), (40, 9, 11), (24, 140, 110)], False),
                                           ([(4, 8, 1)], True)])
def test_failed_allocations_are_reported_before_any_launch(tmp_path, meshes, single):
    _run(tmp_path, FAILURES, meshes=meshes, single=single)


@pytest.mark.skipif((os.cpu_count() or 1) < 8, reason="copies are staged by four threads where there are eight")
def test_octants_below_48_mb_make_no_pinned_buffers(tmp_path):
    # 0.1, 16 and 29 MB; 57 MB
    _run(tmp_path, OCTANT, meshes=[((2, 8, 16), 0), ((4, 256, 256), 0), ((8, 256, 256), 0), ((4, 512, 512), 1)])
