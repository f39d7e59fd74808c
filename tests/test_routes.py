"""Which routes the decode calls take, on the CPU: the library's HIP calls go to a stand-in that
allocates host memory, refuses allocations on demand and counts kernel launches (of Q8_0 / Q4_0
rows: quantize + MFMA GEMV two, the VALU GEMV's single pass one). No kernel runs."""
from __future__ import annotations

import os
import subprocess
import sys

import pytest

import dynalm_amd as dq

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

FAKE = r"""
#include <stddef.h>
#include <stdlib.h>
#include <string.h>
int launches, refuse, capturing, relaxed_mallocs;
static int mode;  /* hipStreamCaptureModeGlobal */
typedef struct { unsigned x, y, z; } d3;
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipSetDevice(int d) { return 0; }
int hipDeviceGetAttribute(int* v, int a, int d) { *v = 256; return 0; }
int hipMalloc(void** p, size_t n) {
  if (refuse) { *p = (void*)16; return 2; }
  relaxed_mallocs += mode == 2;
  *p = malloc(n);
  return 0;
}
int hipFree(void* p) { free(p); return 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int k, void* st) { memcpy(d, s, n); return 0; }
int hipMemsetAsync(void* d, int v, size_t n, void* st) { memset(d, v, n); return 0; }
int hipStreamSynchronize(void* s) { return 0; }
int hipDeviceSynchronize(void) { return 0; }
int hipStreamIsCapturing(void* s, int* c) { *c = capturing; return 0; }
int hipThreadExchangeStreamCaptureMode(int* m) { int o = mode; mode = *m; *m = o; return 0; }
int hipFuncSetAttribute(const void* f, int a, int v) { return 0; }
int hipGetLastError(void) { return 0; }
int __hipPushCallConfiguration(d3 g, d3 b, size_t l, void* s) { return 0; }
int __hipPopCallConfiguration(d3* g, d3* b, size_t* l, void** s) { return 0; }
int hipLaunchKernel(const void* f, d3 g, d3 b, void** a, size_t l, void* s) { ++launches; return 0; }
"""

CALLS = r"""
import ctypes, sys
import numpy as np
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import dynalm_amd as dq
var = lambda n: ctypes.c_int.in_dll(fake, n)
STREAM = 0x1000
def count(w, m, stream=STREAM, **kw):
    for k, v in kw.items(): var(k).value = v
    var("launches").value = 0
    dq.matmul(w, 64, m, w.k, 64, w.n, None, stream)  # (the pointers are never read here)
    for k in kw: var(k).value = 0
    return var("launches").value
def weight(t, n, k):
    return dq.Weight.upload(t, np.zeros((n, dq.row_bytes(t, k)), np.uint8), k)
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    d = tmp_path_factory.mktemp("fakehip")
    (d / "f.c").write_text(FAKE)
    so = str(d / "libfakehip.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-w", "-o", so, str(d / "f.c")], check=True)

    def run(body: str) -> None:
        r = subprocess.run([sys.executable, "-c", CALLS + body, so], cwd=ROOT, capture_output=True, text=True)
        assert r.returncode == 0, r.stdout + r.stderr

    if not os.path.exists(dq.lib_path()):
        pytest.skip("the library is not built")
    return run


def test_without_a_workspace(fake):
    """A refused allocation leaves the call on the GEMV that needs none; a later one gets it."""
    fake("""
w = weight(dq.Q4_0, 300, 512)
assert count(w, 8, refuse=1) == 1
assert count(w, 8, refuse=1) == 1
assert count(w, 8) == 2
assert count(w, 8, refuse=1) == 2  # (it is there now)
assert count(w, 8, capturing=1) == 1
""")


def test_per_thread_default_stream(fake):
    """hipStreamPerThread is one handle for a stream of each thread's own: no buffer is kept for it."""
    fake("""
w = weight(dq.Q8_0, 300, 512)
assert count(w, 8, stream=2) == 1
assert count(w, 8) == 2 and count(w, 8, stream=0) == 2
assert count(w, 8, stream=2) == 1
""")


def test_allocates_in_relaxed_capture_mode(fake):
    """Another thread's capture is neither an obstacle to the allocation nor invalidated by it."""
    fake("""
w = weight(dq.Q4_0, 300, 512)
before = var("relaxed_mallocs").value
assert count(w, 8) == 2 and var("relaxed_mallocs").value == before + 1
m = ctypes.c_int(0)
fake.hipThreadExchangeStreamCaptureMode(ctypes.byref(m))
assert m.value == 0
# a stream that captures itself keeps the mode that refuses: its graph would outlive the buffer
wk = weight(dq.Q4_K, 300, 512)
before = var("relaxed_mallocs").value
var("capturing").value = 1
dq.gemm(wk, dq.ACT_PER32, 64, 64, 0, wk.n, 64, wk.n, None, 0x2000)
assert var("relaxed_mallocs").value == before
""")


def test_where_two_launches_pay(fake):
    """Short rows and few of them stay on one launch of the VALU GEMV (rows32_pays)."""
    fake("""
for t in (dq.Q8_0, dq.Q4_0):
    for n, k, rows in ((300, 512, {2: 1, 3: 1, 4: 1, 5: 2, 7: 2, 8: 2, 12: 2}), (300, 128, {3: 1, 8: 1, 9: 2}),
                       (4096, 4096, {3: 1, 4: 2}), (11008, 4096, {3: 1, 4: 1, 5: 2, 8: 2})):
        w = weight(t, n, k)
        for m, want in rows.items():
            assert count(w, m) == want, (n, k, m)
""")


def test_one_row_jobs_grouped(fake):
    """matmul_many's one-row K-quant jobs share a launch unless their weights fill the CUs alone."""
    fake("""
def many(ws):
    var("launches").value = 0
    dq.matmul_many([(w, 64, 1, w.k, 64, w.n, None) for w in ws], STREAM)
    return var("launches").value
for t in (dq.Q4_K, dq.Q6_K):
    small, wide = weight(t, 500, 512), weight(t, 256 * 64 + 1, 512)
    assert many([small] * 3) == 1 and many([weight(t, 256 * 64, 512)] * 8) == 1
    assert many([wide] * 3) == 3 and many([small, wide, small]) == 2
slab = weight(dq.Q4_K, 9000, 2048)  # two rounds together, one each on the 56-row GEMV
assert many([slab] * 2) == 2 and many([slab] * 3) == 1
assert many([weight(dq.Q4_K, 4096, 2048)] * 2) == 1 and many([weight(dq.Q6_K, 9000, 2048)] * 2) == 1
""")


def test_int16_rows_quantized_in_the_gemv(fake):
    """int16 decode rows are quantized inside the GEMV (one launch less) while rows x weights are few."""
    fake("""
def act(w, m):
    var("launches").value = 0
    dq.matmul_act(w, dq.ACT_Q16, 64, m, w.k, 64, w.n, None, STREAM)
    return var("launches").value
for t, n, k, rows in ((dq.Q4_K, 14336, 512, {1: 1, 4: 1}), (dq.Q6_K, 14336, 512, {1: 1, 2: 1}),
                      (dq.Q4_K, 6144, 14336, {1: 2, 2: 2, 3: 3, 4: 3}), (dq.Q6_K, 14336, 8192, {1: 1, 2: 2})):
    w = weight(t, n, k)
    for m, want in rows.items():
        assert act(w, m) == want, (n, k, m, act(w, m))
""")
