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
