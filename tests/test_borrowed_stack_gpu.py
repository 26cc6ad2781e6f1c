"""8-bit stacks borrowed from memory that starts at any byte, composited without their last frame:
the room behind the selection lets the tiles with wide loads run, on the packed-byte and the exchange
tiles.  Against the oracle, statistics included."""
import numpy as np
import pytest

import chrono_photo_amd as cpa
import oracle_py as O
from chrono_photo_amd import hip as H
from test_parity_gpu import assert_same, make_stack

pytestmark = pytest.mark.gpu


def _borrow(ctx, x, shift):
    n, h, w, c = x.shape
    buf = H.DeviceBuffer(x.nbytes + shift)
    H.check(H.hip().hipMemcpy(buf.ptr + shift, x.ctypes.data, x.nbytes, H.hipMemcpyHostToDevice), "hipMemcpy")
    return buf, cpa.Stack(ctx, w, h, c, 1, device_ptr=buf.ptr + shift, n_frames=n)


@pytest.mark.parametrize("n,s", [(5, 0), (16, 0), (32, 0), (33, 0), (64, 0), (100, 0), (300, 0), (700, 0), (40, 10),
                                 (200, 60), (200, 100)])
@pytest.mark.parametrize("shift", [0, 1, 2, 3])
@pytest.mark.parametrize("c", [1, 2, 3, 4])
def test_any_start_byte(ctx, c, shift, n, s):
    x = np.ascontiguousarray(make_stack(9000 + n + c, n + 1, 5, 27, c, outlier_frac=0.1))
    buf, st = _borrow(ctx, x, shift)
    sample = sorted(np.random.default_rng(n).choice(n, s, replace=False).tolist()) if s else None
    for absolute, lo, hi, bg, sel in ((True, 0.05, 0.2, 0, 2), (False, 2.0, 4.0, 2, 3)):
        proc = cpa.OutlierProcessor(cpa.Threshold(absolute, lo, hi), bg, sel, sample_indices=sample)
        img, mask, stats = proc.process(st, image_indices=range(n), with_stats=True)
        oimg, omask, owarn, ost = O.outlier(x, O.threshold(absolute, lo, hi, 1), bg, sel, slots=list(range(n)),
                                            sample_pos=sample, stats=True)
        assert_same((img, mask, stats, proc.warnings), (oimg, omask, ost, owarn), f"{c} {shift} {n} {s} {absolute}")
    st.close()
    buf.free()
