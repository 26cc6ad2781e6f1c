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


@pytest.mark.parametrize("n", [40, 100, 200, 300, 500])
@pytest.mark.parametrize("c,margin", [(1, 9), (1, 11), (2, 5), (2, 7)])
def test_narrow_margin_keeps_a_tile(ctx, c, margin, n):
    """The last frame's last row with less room behind it than the exchange tiles' four-pixel loads
    need and enough for one pixel's: the one-pixel tiles of the same frame counts take it (a job on
    the generic kernel would not be grouped)."""
    w, out_w, h = 40, 29, 5
    x = np.ascontiguousarray(make_stack(9300 + n + c, n, h, w, c, outlier_frac=0.1))
    buf, st = _borrow(ctx, x, 0)
    origin = np.tile(np.array([[w - out_w - margin, 0]], np.int32), (n, 1))
    px, mask = H.DeviceBuffer(out_w * h * c), H.DeviceBuffer(out_w * h * c)
    for absolute, lo, hi, bg, sel in ((True, 0.05, 0.2, 0, 2), (False, 2.0, 4.0, 2, 3)):
        proc = cpa.OutlierProcessor(cpa.Threshold(absolute, lo, hi), bg, sel)
        batch = cpa.Batch(ctx, [cpa.Job(cpa.CP_MODE_OUTLIER, st, px.ptr, mask.ptr, processor=proc, crop=(origin, out_w, h))])
        assert batch.info()["group_jobs"] == 1, batch.info()
        batch.launch()
        ctx.synchronize()
        oimg, omask, _ = O.outlier(x, O.threshold(absolute, lo, hi, 1), bg, sel, crop_xy=origin, out_w=out_w, out_h=h)
        assert np.array_equal(px.to_host(np.zeros((h, out_w, c), np.uint8)), oimg)
        assert np.array_equal(mask.to_host(np.zeros((h, out_w, c), np.uint8)), omask)
        batch.close()
    st.close()
    for b in (buf, px, mask):
        b.free()
