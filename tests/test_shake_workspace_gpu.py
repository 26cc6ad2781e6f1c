"""The workspace cp_shake keeps with its context: not on a context with a device-memory budget, and not
needed where there is no room for it."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

import chrono_photo_amd as cpa
from chrono_photo_amd import hip as H

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _free_bytes():
    free, total = C.c_size_t(), C.c_size_t()
    H.check(H.hip().hipMemGetInfo(C.byref(free), C.byref(total)), "hipMemGetInfo")
    return free.value


def test_a_budgeted_context_keeps_no_device_memory(ctx):
    x = np.random.default_rng(5).integers(0, 256, (4, 32, 40, 3), np.uint8)

    def search(c):
        st = cpa.Stack.from_array(c, x)
        cpa.SimpleProcessor().process(st)
        before = _free_bytes()
        off = cpa.ShakeAnalyzer().analyze(st, [(20, 16)], 4, 3)
        after = _free_bytes()
        st.close()
        return off, before - after

    ref, _ = search(ctx)  # the kernels are loaded with the first call of a process
    small = cpa.Context(0, hbm_budget=1 << 20)
    off, kept = search(small)
    small.close()
    assert np.array_equal(off, ref)
    assert kept == 0, kept


# Fails the workspace's allocation (its size alone) with the runtime's own out-of-memory error.
NO_WORKSPACE = r"""
#include <dlfcn.h>
#include <stddef.h>
typedef int (*malloc_fn)(void**, size_t);
extern "C" int hipMalloc(void** p, size_t n) {
    void* h = dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD);
    malloc_fn real = (malloc_fn)dlsym(h, "hipMalloc");
    return real(p, n == (size_t)4 << 20 ? (size_t)1 << 50 : n);
}
"""

SEARCH = r'''
import ctypes, sys
ctypes.CDLL(sys.argv[2], mode=ctypes.RTLD_GLOBAL)
sys.path[:0] = [sys.argv[1]]
import numpy as np
import chrono_photo_amd as cpa
print("case: shake search whose workspace cannot be allocated", flush=True)
x = np.random.default_rng(5).integers(0, 256, (4, 32, 40, 3), np.uint8)
ctx = cpa.Context(0)
st = cpa.Stack.from_array(ctx, x)
off = cpa.ShakeAnalyzer().analyze(st, [(20, 16)], 4, 3)
print("OFFSETS", off.reshape(-1).tolist(), flush=True)
'''


def test_search_without_room_for_the_workspace(ctx, tmp_path):
    """The smaller allocations of the call itself still succeed, and so does the call."""
    (tmp_path / "no_ws.cpp").write_text(NO_WORKSPACE)
    lib = str(tmp_path / "no_ws.so")
    subprocess.run(["g++", "-shared", "-fPIC", "-o", lib, str(tmp_path / "no_ws.cpp"), "-ldl"], check=True)
    r = subprocess.run([sys.executable, "-c", SEARCH, os.path.join(ROOT, "chrono-photo_amd"), lib],
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
    x = np.random.default_rng(5).integers(0, 256, (4, 32, 40, 3), np.uint8)
    st = cpa.Stack.from_array(ctx, x)
    ref = cpa.ShakeAnalyzer().analyze(st, [(20, 16)], 4, 3)
    st.close()
    assert f"OFFSETS {ref.reshape(-1).tolist()}" in r.stdout


def test_an_error_before_the_search_is_reported(ctx):
    """An error that an earlier runtime call left unread ends the call, as it ends a composite, and is
    gone with it; it never stands for offsets that were not written."""
    x = np.random.default_rng(6).integers(0, 256, (4, 32, 40, 3), np.uint8)
    st = cpa.Stack.from_array(ctx, x)
    ref = cpa.ShakeAnalyzer().analyze(st, [(20, 16)], 4, 3)
    assert ref.any()
    p = C.c_void_p()
    assert H.hip().hipMalloc(C.byref(p), 1 << 50) != 0
    with pytest.raises(cpa.ChronoError) as e:
        cpa.ShakeAnalyzer().analyze(st, [(20, 16)], 4, 3)
    assert e.value.code == cpa.CP_ERR_HIP
    assert np.array_equal(cpa.ShakeAnalyzer().analyze(st, [(20, 16)], 4, 3), ref)
    st.close()
