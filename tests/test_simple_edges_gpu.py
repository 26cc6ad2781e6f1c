"""Darker / lighter at the ends of rows: rows and whole frames that end inside a lane's pixels, from one
wave to several per row, with the frames' offsets from their spacing and from a table.  Against the
oracle, bit-exact."""
import numpy as np
import pytest

import chrono_photo_amd as cpa
import oracle_py as O
from test_parity_gpu import make_stack

pytestmark = pytest.mark.gpu

FADE = (False, True, [(0, 0.3), (9, 1.0)])


def _check(x, st, msg, slots=None, crop=None):
    oc = {} if crop is None else dict(crop_xy=crop[0], out_w=crop[1], out_h=crop[2])
    for weights, fade, darker in (((1, 1, 1, 1), None, True), ((1, 1, 1, 1), None, False),
                                  ((0.5, 1, 0.3, 2), None, False), ((1, 1, 1, 1), FADE, True)):
        img = cpa.SimpleProcessor(weights, cpa.Fade.none() if fade is None else cpa.Fade(*fade), darker).process(
            st, crop=crop, image_indices=slots)
        ofade = O.Fade.none() if fade is None else O.Fade(fade[0], fade[1], [f for f, _ in fade[2]], [v for _, v in fade[2]])
        ref = O.simple(x, weights, ofade, darker, slots=slots, **oc)
        assert np.array_equal(img, ref), (msg, weights, darker)


@pytest.mark.parametrize("bits,c", [(8, 1), (8, 2), (8, 3), (8, 4), (16, 1), (16, 2), (16, 3), (16, 4)])
@pytest.mark.parametrize("w,h", [(129, 5), (131, 2), (133, 3), (16, 16), (17, 15), (257, 1), (515, 2)])
def test_whole_frames(ctx, bits, c, w, h):
    """One row of w * h pixels; evenly spaced frames forward and backward, uneven ones."""
    n = 12
    x = make_stack(w * h + c, n, h, w, c, bits=bits, outlier_frac=0.3)
    st = cpa.Stack.from_array(ctx, x)
    for slots in (None, list(range(n))[::-1], [0, 1, 2, 4, 5, 7, 8, 10, 11]):
        _check(x, st, (bits, c, w, h, slots), slots=slots)
    st.close()


@pytest.mark.parametrize("bits,c", [(8, 1), (8, 2), (8, 3), (8, 4), (16, 1), (16, 2), (16, 3), (16, 4)])
@pytest.mark.parametrize("w", [126, 127, 128, 129, 131, 253, 255, 256, 257, 258, 259, 260, 515])
def test_cropped_rows(ctx, bits, c, w):
    """Rows of w pixels out of w + 3; the same origin for every frame, different ones, and crops
    that keep the full width."""
    n, h = 11, 6
    x = make_stack(w + c, n, h, w + 3, c, bits=bits, outlier_frac=0.3)
    st = cpa.Stack.from_array(ctx, x)
    rng = np.random.default_rng(w)
    same = np.tile(np.array([[1, 2]], np.int32), (n, 1))
    mixed = rng.integers(0, (4, 3), (n, 2)).astype(np.int32)
    _check(x, st, (bits, c, w, "same"), crop=(same, w, h - 2))
    _check(x, st, (bits, c, w, "mixed"), crop=(mixed, w, h - 2))
    vertical = np.stack([np.zeros(n, np.int32), rng.integers(0, 3, n).astype(np.int32)], 1)
    _check(x, st, (bits, c, w, "vertical"), crop=(vertical, w + 3, h - 2))
    st.close()


@pytest.mark.parametrize("c", [3, 4])
@pytest.mark.parametrize("w,h", [(1600, 655), (1439, 729), (1600, 983), (1921, 819), (1601, 1309), (2048, 1024)])
def test_large_whole_frames(ctx, c, w, h):
    """8-bit images of about half, three quarters and all of what the device holds at once, one frame
    more than the loads in flight."""
    n = 9
    x = np.random.default_rng(w + h + c).integers(0, 256, (n, h, w, c), dtype=np.uint8)
    st = cpa.Stack.from_array(ctx, x)
    for darker in (True, False):
        img = cpa.SimpleProcessor((1, 1, 1, 1), cpa.Fade.none(), darker).process(st)
        assert np.array_equal(img, O.simple(x, (1, 1, 1, 1), O.Fade.none(), darker)), (c, w, h, darker)
    st.close()
