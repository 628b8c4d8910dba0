"""Device errors in the network's training and gradient calls reach the caller.

A small host library stands in for the HIP runtime in a child process: device
memory is host memory, kernels do nothing, and the n-th wait or the n-th copy
back from the device fails on request. No GPU is involved.
"""
from __future__ import annotations

import os
import subprocess
import sys

import pytest

from common import ROOT

RUNTIME = r"""
#include <cstdlib>
#include <cstring>
extern "C" {
int fail_wait = 0, fail_copy = 0;  // countdown to the call that fails (0: none)
static int down(int &n) { return n > 0 && --n == 0 ? 999 : 0; }
int hipGetDeviceCount(int *n) { *n = 1; return 0; }
int hipGetDevice(int *d) { *d = 0; return 0; }
int hipDeviceGetAttribute(int *v, int, int) { *v = 8; return 0; }
int hipGetLastError() { return 0; }
int hipMalloc(void **p, size_t n) { *p = std::calloc(n ? n : 1, 1); return *p ? 0 : 2; }
int hipFree(void *p) { std::free(p); return 0; }
int hipMemset(void *p, int v, size_t n) { std::memset(p, v, n); return 0; }
int hipMemsetAsync(void *p, int v, size_t n, void *) { std::memset(p, v, n); return 0; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *) {
    if (kind == 2 && down(fail_copy)) return 999;
    std::memcpy(d, s, n);
    return 0;
}
int hipStreamCreateWithFlags(void **s, unsigned) { *s = std::malloc(1); return 0; }
int hipStreamDestroy(void *s) { std::free(s); return 0; }
int hipStreamSynchronize(void *) { return down(fail_wait); }
int hipStreamWaitEvent(void *, void *, unsigned) { return 0; }
int hipEventCreateWithFlags(void **e, unsigned) { *e = std::malloc(1); return 0; }
int hipEventDestroy(void *e) { std::free(e); return 0; }
int hipEventRecord(void *, void *) { return 0; }
struct dim { unsigned x, y, z; };
int __hipPushCallConfiguration(dim, dim, size_t, void *) { return 0; }
int __hipPopCallConfiguration(dim *, dim *, size_t *, void **) { return 0; }
int hipLaunchKernel(const void *, dim, dim, void **, size_t, void *) { return 0; }
}
"""

CHILD = r"""
import ctypes as C, sys
import numpy as np
rt = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)  # ahead of the runtime that the library links
from thor_amd import capi
hidden, call, what, nth = int(sys.argv[2]), sys.argv[3], sys.argv[4], int(sys.argv[5])
fail = C.c_int.in_dll(rt, what)
m = capi.MLP(9, hidden, 4)
X, Y = np.ones((70, 9), np.float32), np.ones((70, 4), np.float32)
m.set_data(X, Y)
run = (lambda: m.train_epoch(32, 1e-3, 0)) if call == "epoch" else (lambda: m.gradients(X, Y))
run()  # buffers are in place: the calls that follow wait and copy for their results only
fail.value = nth
try:
    run()
except capi.ThorError as e:
    assert e.code == capi.THOR_ERR_HIP, e
    assert fail.value == 0
    run()  # the error was the call's own
    print("raised")
else:
    print("returned")
"""


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    d = tmp_path_factory.mktemp("runtime")
    src, lib = d / "runtime.cpp", d / "libruntime.so"
    src.write_text(RUNTIME)
    subprocess.run(["g++", "-shared", "-fPIC", "-O1", "-o", str(lib), str(src)], check=True)
    return str(lib)


# the fused form (256 hidden units) reads the epoch's errors back once, the
# layer-by-layer form each batch's (here three); thor_mlp_gradients copies and
# waits for the gradients, then for the loss
@pytest.mark.parametrize("hidden,call,nth", [(256, "epoch", 1), (64, "epoch", 1), (64, "epoch", 3),
                                             (256, "gradients", 1), (256, "gradients", 2), (64, "gradients", 2)])
@pytest.mark.parametrize("what", ["fail_wait", "fail_copy"])
def test_device_error_is_returned(built, runtime, hidden, call, what, nth):
    r = subprocess.run([sys.executable, "-c", CHILD, runtime, str(hidden), call, what, str(nth)], cwd=ROOT,
                       env=dict(os.environ, PYTHONPATH=ROOT), capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.split()[-1] == "raised", r.stdout + r.stderr
