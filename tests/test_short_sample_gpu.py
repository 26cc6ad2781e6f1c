"""`--sample` on 16-bit stacks of a few frames, at both sides of the line between the generic kernel and
the tiles with a sample block, against the oracle."""

import numpy as np
import pytest

from test_partial_tiles_gpu import CASES, _stack, assert_same, run_both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,s", [(3, 3), (4, 3), (9, 9), (10, 4), (10, 5), (11, 3), (11, 7), (11, 8), (15, 3), (16, 3),
                                 (16, 16)])
@pytest.mark.parametrize("c", [1, 2, 3, 4])
def test_u16_short_samples(ctx, n, s, c):
    x = _stack(9900 + 31 * n + s + c, n, c, 16)
    sample = sorted(np.random.default_rng(n + s).choice(n, s, replace=False).tolist())
    for absolute, lo, hi, bg, sel, weights in CASES:
        gpu, ref = run_both(ctx, x, absolute, lo, hi, bg, sel, weights=weights, sample=sample)
        assert_same(gpu, ref, f"n={n} s={s} c={c} abs={absolute} bg={bg} sel={sel} w={weights}")
