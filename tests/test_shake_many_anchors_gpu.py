"""Shake searches whose workgroups need more than one launch (65535 rows of a grid each), and the
number of anchors at which a call is refused."""
import numpy as np
import pytest

import chrono_photo_amd as cpa
import oracle_py as O

pytestmark = pytest.mark.gpu


def _case(bits, c, r, s, n_anchors):
    rng = np.random.default_rng(n_anchors + r)
    w, h = 2 * (r + s) + 20, 2 * (r + s) + 13
    x = rng.integers(0, 1 << bits, (3, h, w, c)).astype(np.uint8 if bits == 8 else np.uint16)
    m = r + s
    anchors = np.stack([rng.integers(m, w - m, n_anchors), rng.integers(m, h - m, n_anchors)], 1)
    return x, anchors.astype(np.int32)


@pytest.mark.parametrize("bits,c,r,s,n_anchors", [(8, 1, 8, 1, 40000),    # two window chunks: 80000 groups
                                                   (16, 1, 8, 1, 33000),
                                                   (8, 3, 0, 17, 20000)])  # four candidate blocks
def test_more_than_one_launch(ctx, bits, c, r, s, n_anchors):
    x, anchors = _case(bits, c, r, s, n_anchors)
    st = cpa.Stack.from_array(ctx, x)
    off = cpa.ShakeAnalyzer().analyze(st, anchors, r, s)
    st.close()
    assert np.array_equal(off, O.shake(x, anchors, r, s))


def test_too_many_anchors_are_refused(ctx):
    x, anchors = _case(8, 1, 1, 1, 65536)
    st = cpa.Stack.from_array(ctx, x)
    with pytest.raises(cpa.ChronoError) as e:
        cpa.ShakeAnalyzer().analyze(st, anchors, 1, 1)
    st.close()
    assert e.value.code == cpa.CP_ERR_INVALID_ARG
