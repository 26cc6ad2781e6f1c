"""8-bit tiles whose lanes exchange the dwords they load, and the ranks read from bit planes:
partial counts of each tile, widths that end inside the four pixels of a load, crops, frame
selections with even steps (forward, backward) and without, and the `--sample` block.  Results
are whole numbers or the oracle's own float steps in its order, so everything is compared for
equality, statistics included."""
import numpy as np
import pytest

import chrono_photo_amd as cpa
from test_parity_gpu import assert_same, make_stack, run_both

pytestmark = pytest.mark.gpu

# bucket, tile, frame counts: the tile full, one short, one past a lane's block
TILES = [(2, (1, 64, 4, 1), (33, 63, 64)), (3, (2, 64, 4, 1), (65, 127, 128)), (4, (4, 64, 4, 1), (129, 193, 256)),
         (5, (8, 64, 4, 1), (257, 449, 512)), (6, (8, 96, 4, 1), (513, 577, 768)), (7, (8, 128, 4, 1), (769, 897, 1024)),
         (8, (8, 160, 4, 1), (1025, 1121, 1279))]
# absolute, min, max, background, outlier: every background (1 draws frames), first / extreme /
# average / forward / backward outliers
MODES = [(True, 0.05, 0.2, 0, 2), (True, 0.02, 0.2, 2, 3), (True, 0.0, 0.1, 1, 4), (False, 2.0, 4.0, 3, 5),
         (False, 0.5, 2.0, 2, 3), (False, 1.5, 3.0, 0, 1)]


def _selections(n_stack, n):
    rng = np.random.default_rng(n)
    uneven = np.sort(rng.choice(n_stack, n, replace=False))
    return [None, np.arange(n)[::-1], uneven]


@pytest.mark.parametrize("bucket,tile,counts", TILES)
@pytest.mark.parametrize("c", [1, 2, 3, 4])
def test_exchange_tiles(ctx, bucket, tile, counts, c):
    shapes = [None] * len(cpa.TILE_BUCKETS)
    shapes[bucket] = tile
    cpa.tile_shapes_set(ctx, 1, c, shapes)
    try:
        for i, n in enumerate(counts):
            w = (21, 38, 67)[i]
            x = make_stack(8000 + n + c, n + 3, 4, w, c, outlier_frac=0.4 if i == 0 else 0.06)
            sel = _selections(n + 3, n)[i]
            slots = (list(range(n)) if sel is None else sel.tolist())
            crop = None
            if i == 1:
                offs = np.stack([np.arange(n) % 3, np.arange(n) % 2], 1).astype(np.int32)
                crop = (offs, w - 3, 3)
            for mode in MODES:
                gpu, ref = run_both(ctx, x, *mode, slots=slots, crop=crop, seed=11)
                assert_same(gpu, ref, f"{tile} n={n} c={c} mode={mode}")
    finally:
        cpa.tile_shapes_set(ctx, 1, c, [])


@pytest.mark.parametrize("n,s", [(200, 1), (256, 128), (257, 65), (512, 127), (513, 17), (1280, 128)])
@pytest.mark.parametrize("c", [1, 2, 3, 4])
def test_exchange_sample_block(ctx, n, s, c):
    x = make_stack(8300 + n + s + c, n, 4, 23, c, outlier_frac=0.1)
    sample = sorted(np.random.default_rng(n + s).choice(n, s, replace=False).tolist())
    for mode in MODES:
        if not mode[0] and s < 3:  # relative thresholds need three samples
            continue
        gpu, ref = run_both(ctx, x, *mode, sample=sample, seed=3)
        assert_same(gpu, ref, f"n={n} s={s} c={c} mode={mode}")


def _plane_stack(seed, n, c, bits):
    """Rows of different order statistics: all bits random, few distinct values, two values at
    neighbouring powers of two, the ends of the range, constant."""
    rng = np.random.default_rng(seed)
    top = (1 << bits) - 1
    x = rng.integers(0, top + 1, (n, 6, 19, c))
    x[:, 1] = rng.integers(0, 3, (n, 19, c)) * (top // 3)
    x[:, 2] = (1 << (bits - 1)) - rng.integers(0, 2, (n, 19, c))
    x[:, 3] = np.where(rng.random((n, 19, c)) < 0.5, 0, top)
    x[:, 4] = top - rng.integers(0, 2, (n, 19, c))
    x[:, 5] = rng.integers(0, top + 1, (1, 19, c))
    return x.astype(np.uint8 if bits == 8 else np.uint16)


PLANES = [(8, 1, (1, 32, 1, 1), (17, 32)), (8, 2, (1, 64, 1, 1), (33, 64)), (8, 2, (2, 32, 1, 1), (50, 64)),
          (8, 5, (16, 32, 1, 1), (300, 511)), (8, 6, (8, 96, 4, 1), (600, 768)),
          (16, 1, (1, 32, 2), (17, 32)), (16, 1, (1, 32, 1), (31, 32)), (16, 3, (4, 32, 2), (65, 128)),
          (16, 4, (8, 32, 2), (129, 256)), (16, 4, (8, 32, 1), (200, 255)), (16, 5, (16, 32, 2), (257, 512)),
          (16, 5, (8, 64, 1), (400, 512))]


@pytest.mark.parametrize("bits,bucket,tile,counts", PLANES)
@pytest.mark.parametrize("c", [3, 4])
def test_bit_plane_ranks(ctx, bits, bucket, tile, counts, c):
    shapes = [None] * len(cpa.TILE_BUCKETS)
    shapes[bucket] = tile
    cpa.tile_shapes_set(ctx, bits // 8, c, shapes)
    try:
        for n in counts:
            x = _plane_stack(8600 + n + c, n, c, bits)
            for mode in ((False, 0.5, 2.0, 0, 2), (False, 2.0, 4.0, 2, 3), (True, 0.05, 0.2, 3, 2)):
                gpu, ref = run_both(ctx, x, *mode)
                assert_same(gpu, ref, f"{bits} {tile} n={n} c={c} mode={mode}")
    finally:
        cpa.tile_shapes_set(ctx, bits // 8, c, [])


@pytest.mark.parametrize("n", [257, 300, 700, 1024])
@pytest.mark.parametrize("c", [1, 3])
def test_u16_sums_past_24_bits(ctx, n, c):
    """Averages over more than 256 frames near the top of the range, whose f32 sums round."""
    rng = np.random.default_rng(n + c)
    x = rng.integers(60000, 65536, (n, 3, 21, c)).astype(np.uint16)
    x[rng.random((n, 3, 21)) < 0.1] = 3
    for mode in ((True, 0.3, 0.5, 2, 3), (True, 0.02, 0.1, 2, 2), (False, 1.0, 2.0, 2, 3)):
        gpu, ref = run_both(ctx, x, *mode)
        assert_same(gpu, ref, f"n={n} c={c} mode={mode}")


@pytest.mark.parametrize("c", [3, 4])
def test_u16_batch_group_to_512_frames(ctx, c):
    """16-bit 3/4-channel jobs of 257 to 512 frames share a group launch, absolute thresholds on the
    two-pixel tile and relative ones on the one-pixel tile; widths inside a pixel pair."""
    import oracle_py as O
    from chrono_photo_amd import hip as H
    jobs, keep = [], []
    for i, (n, w) in enumerate(((257, 33), (300, 40), (449, 18), (512, 35))):
        x = make_stack(8800 + n + c, n, 5, w, c, bits=16, outlier_frac=0.1)
        st = cpa.Stack.from_array(ctx, x)
        thr = cpa.Threshold.abs(0.05, 0.2) if i % 2 == 0 else cpa.Threshold.rel(2.0, 4.0)
        px, mask = H.DeviceBuffer(x[0].nbytes), H.DeviceBuffer(x[0].size)
        jobs.append(cpa.Job(cpa.CP_MODE_OUTLIER, st, px.ptr, mask.ptr, processor=cpa.OutlierProcessor(thr, i, i + 1, seed=3)))
        keep.append((x, st, px, mask))
    batch = cpa.Batch(ctx, jobs, graph=True)
    info = batch.info()
    assert info["group_jobs"] == 4 and info["group_launches"] == 2, info
    for rep in range(3):
        batch.launch()
        ctx.synchronize()
        for i, (x, st, px, mask) in enumerate(keep):
            lo, hi = ((0.05, 0.2), (2.0, 4.0))[i % 2]
            oimg, omask, _ = O.outlier(x, O.threshold(i % 2 == 0, lo, hi, 2), i, i + 1, seed=3)
            assert np.array_equal(px.to_host(np.zeros(x[0].shape, x.dtype)), oimg), (rep, i)
            assert np.array_equal(mask.to_host(np.zeros(x[0].shape, np.uint8)), omask), (rep, i)
    batch.close()
    for x, st, px, mask in keep:
        st.close()
        px.free()
        mask.free()
