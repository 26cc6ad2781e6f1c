"""Outlier tiles that the stack does not fill: frame counts one past a lane block, one short of a
tile and in between, where the lanes' pads must neither count as outliers nor be a lane's largest
distance.  Thresholds go down to zero, where every frame (and any pad) passes the test, and the
samples include pixels whose frames all sit at the median, so that pads tie with frames.
Bit-exact against the oracle, statistics included."""
import numpy as np
import pytest

import chrono_photo_amd as cpa
from test_parity_gpu import assert_same, make_stack, run_both
from test_u8_kernel_gpu import U8_CHOICES

pytestmark = pytest.mark.gpu

# (n): around the lane blocks and tiles of the 8-bit shapes
COUNTS8 = [4, 15, 17, 33, 60, 63, 65, 97, 127, 129, 250, 257, 500, 513, 700, 769, 1000, 1025, 1200, 1279]


def _stack(seed, n, c, bits):
    x = make_stack(seed, n, 5, 23, c, bits=bits, outlier_frac=0.1)
    top = (1 << bits) - 1
    x[:, 1, 2:9, :] = 77                                    # every frame at the median
    x[:, 2, 2:9, :] = 40 + (np.arange(n) % 2)[:, None, None]  # half-way medians
    x[:, 3, 2:9, :] = np.where(np.arange(n) % 3 == 0, top, 0)[:, None, None]  # the ends of the range
    return x


CASES = ((True, 0.05, 0.2, 0, 2, (1, 1, 1, 1)), (True, 0.0, 0.1, 3, 2, (1, 1, 1, 1)), (True, 0.02, 0.2, 2, 3, (1, 1, 1, 1)),
         (False, 0.0, 2.0, 0, 2, (1, 1, 1, 1)), (False, 2.0, 4.0, 2, 4, (1, 1, 1, 1)), (True, 0.04, 0.1, 1, 5, (0.5, 1, 0, 1)),
         (False, 1.0, 2.0, 0, 2, (1, -0.5, 1, 1)), (True, 0.0, 0.05, 0, 1, (-1, 1, 1, 1)))


def _check(ctx, x, msg):
    for absolute, lo, hi, bg, sel, weights in CASES:
        gpu, ref = run_both(ctx, x, absolute, lo, hi, bg, sel, weights=weights)
        assert_same(gpu, ref, f"{msg} abs={absolute} lo={lo} bg={bg} sel={sel} w={weights}")


@pytest.mark.parametrize("n", COUNTS8)
@pytest.mark.parametrize("c", [1, 2, 3, 4])
def test_u8_partial_tiles(ctx, n, c):
    """The packed-byte kernel, pinned where a bucket's default is another one."""
    x = _stack(9100 + 7 * n + c, n, c, 8)
    cpa.tile_shapes_set(ctx, 1, c, U8_CHOICES[0])
    try:
        _check(ctx, x, f"n={n} c={c}")
    finally:
        cpa.tile_shapes_set(ctx, 1, c, [])


COUNTS16 = [3, 15, 17, 31, 33, 63, 65, 100, 129, 255, 257, 300, 511, 513, 700, 1023, 1024, 1025]


@pytest.mark.parametrize("n", COUNTS16)
@pytest.mark.parametrize("c", [1, 2, 3, 4])
def test_u16_partial_tiles(ctx, n, c):
    """16-bit tiles of two or four pixels per lane, 1-32 lanes per group, and the widths that end
    inside a lane's pixels; above 1024 frames, and for averages above 256, the generic kernel."""
    _check(ctx, _stack(9500 + 7 * n + c, n, c, 16), f"n={n} c={c}")


@pytest.mark.parametrize("n,s", [(40, 5), (100, 48), (128, 64), (128, 65), (200, 128), (256, 3), (300, 48), (512, 128),
                                 (600, 128), (1024, 100), (1024, 129), (1025, 64)])
@pytest.mark.parametrize("c", [1, 2, 3, 4])
def test_u16_sample_subsets(ctx, n, s, c):
    """`--sample` on 16-bit stacks: the ranks from their own block of up to 128 sample frames, the
    distances over all frames."""
    x = _stack(9700 + n + s + c, n, c, 16)
    sample = sorted(np.random.default_rng(n + s).choice(n, s, replace=False).tolist())
    for absolute, lo, hi, bg, sel, weights in CASES:
        gpu, ref = run_both(ctx, x, absolute, lo, hi, bg, sel, weights=weights, sample=sample)
        assert_same(gpu, ref, f"n={n} s={s} c={c} abs={absolute} bg={bg} sel={sel} w={weights}")


@pytest.mark.parametrize("c,n", [(1, 100), (2, 60), (1, 300), (3, 400)])
def test_u16_wrapped_stacks(ctx, c, n):
    """Borrowed 16-bit memory that ends with its last sample: wide loads that would pass the end
    go another way."""
    from chrono_photo_amd import hip as H
    import oracle_py as O
    x = _stack(9900 + n + c, n, c, 16)
    buf = H.DeviceBuffer(x.nbytes)
    buf.from_host(np.ascontiguousarray(x))
    st = cpa.Stack(ctx, x.shape[2], x.shape[1], c, 2, device_ptr=buf.ptr, n_frames=n)
    img, mask = cpa.OutlierProcessor(cpa.Threshold.abs(0.05, 0.2), 0, 2).process(st)
    oimg, omask, _ = O.outlier(x, O.threshold(True, 0.05, 0.2, 2), 0, 2)
    assert np.array_equal(img, oimg) and np.array_equal(mask, omask)
    st.close()
    buf.free()


@pytest.mark.parametrize("r,s", [(0, 0), (1, 7), (5, 8), (7, 15), (10, 16), (21, 20), (32, 12), (3, 33)])
@pytest.mark.parametrize("bits,c", [(8, 1), (8, 3), (16, 1), (16, 2), (16, 3), (16, 4)])
def test_shake_tile_edges(ctx, r, s, bits, c):
    """Candidate blocks of 1, 15-17, 31-33 and more columns, and region rows around whole slabs of
    64 samples, on unstructured frames (every sum distinct)."""
    import oracle_py as O
    rng = np.random.default_rng(100 * r + s + bits + c)
    m = r + s
    h, w = 2 * m + 9, 2 * m + 14
    x = rng.integers(0, 1 << bits, (4, h, w, c)).astype(np.uint8 if bits == 8 else np.uint16)
    x[2] = (1 << bits) - 1
    x[3] = np.where(rng.random((h, w, 1)) < 0.5, 0, (1 << bits) - 1)
    anchors = [(m, m), (w - 1 - m, h - 1 - m)]
    st = cpa.Stack.from_array(ctx, x)
    got = cpa.ShakeAnalyzer().analyze(st, anchors, r, s)
    st.close()
    assert np.array_equal(got, O.shake(x, anchors, r, s))


@pytest.mark.parametrize("bits,c", [(8, 1), (8, 3), (8, 4), (16, 1), (16, 3), (16, 4)])
@pytest.mark.parametrize("darker", [True, False])
@pytest.mark.parametrize("n,w", [(1, 4), (7, 5), (8, 6), (9, 7), (17, 130), (40, 257)])
def test_simple_unit_weights(ctx, bits, c, darker, n, w):
    """Whole-number darker / lighter steps: ties keep the first frame, black and white pixels,
    frame counts around the eight in flight, widths inside a lane's pixels."""
    import oracle_py as O
    rng = np.random.default_rng(n * 31 + w + c)
    top = (1 << bits) - 1
    x = rng.integers(0, top + 1, (n, 5, w, c)).astype(np.uint8 if bits == 8 else np.uint16)
    x[:, 1] = 0
    x[:, 2] = top
    x[:, 3] = np.roll(np.arange(c) * 9 + 5, 1)
    x[::2, 3] = (np.arange(c) * 9 + 5)[::-1]  # the same sum in another order: the first one stays
    st = cpa.Stack.from_array(ctx, x)
    crop = (np.stack([np.arange(n) % 2, np.arange(n) % 3], 1), w - 1, 3)
    for cr in (None, crop):
        img = cpa.SimpleProcessor(darker=darker).process(st, crop=cr)
        ref = O.simple(x, darker=darker, **({} if cr is None else dict(crop_xy=cr[0], out_w=cr[1], out_h=cr[2])))
        assert np.array_equal(img, ref), (bits, c, darker, n, w, cr is not None)
    st.close()
