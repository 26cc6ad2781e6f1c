"""The workspace cp_shake keeps with its context: not on a context with a device-memory budget."""
import ctypes as C

import numpy as np
import pytest

import chrono_photo_amd as cpa
from chrono_photo_amd import hip as H

pytestmark = pytest.mark.gpu


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
