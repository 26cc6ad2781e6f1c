// kernels.hip -- kernel instantiation and launch policy for the compositing modes.
#include "k_outlier_generic.h"
#include "k_simple.h"
#include "kernels_fast.h"
#include "kernels_u8.h"
#include "runtime.h"

namespace cp {

template <int B, int C>
static void launch_outlier_generic_c(const OutlierK& k, hipStream_t s) {
    dim3 block(256), grid((k.out_w + 255) / 256, k.out_h);
    if (k.pos_off.table) hipLaunchKernelGGL((outlier_generic_kernel<B, C, true>), grid, block, 0, s, k);
    else hipLaunchKernelGGL((outlier_generic_kernel<B, C, false>), grid, block, 0, s, k);
}

template <int B>
static void launch_outlier_generic_b(const cp_stack* st, const OutlierK& k, hipStream_t s) {
    switch (st->channels) {
    case 1: launch_outlier_generic_c<B, 1>(k, s); break;
    case 2: launch_outlier_generic_c<B, 2>(k, s); break;
    case 3: launch_outlier_generic_c<B, 3>(k, s); break;
    default: launch_outlier_generic_c<B, 4>(k, s); break;
    }
}

OutlierPlan plan_outlier(cp_ctx* ctx, const cp_stack* st, const OutlierK& k, uint64_t max_pos, uint32_t flags) {
    // 8-bit composites take the packed-byte kernel up to 1280 frames (and, with a `--sample`
    // subset, up to 128 sample frames) or the tuned choice between the two kernels; 16-bit ones
    // the 16-bit kernel up to 1024 frames (and up to 128 sample frames); the one-lane-per-pixel
    // generic kernel takes the rest.  A packed-byte choice whose wide loads would read past a
    // borrowed stack's end falls back to another candidate of its bucket, or to the generic kernel
    // where none stays inside the stack.
    OutlierPlan p;
    const bool sums = k.background == 2 || k.outlier == 3;
    if (flags & CP_FLAG_FORCE_GENERIC) return p;
    auto u8_fits = [&](int sh) {
        return u8_tile_fits(st->dev, st->alloc_bytes, st->channels, kU8Shapes[sh].load_px(), k, max_pos);
    };
    if (k.sample_mask != nullptr) {
        if (st->bps == 1 && k.n <= kU8MaxFrames && k.n_sample <= kU8MaxSample && k.samp_off) {
            int sh = u8_sample_shape(k.n, k.n_sample, true);
            if (sh < 0 || !u8_fits(sh)) sh = u8_sample_shape(k.n, k.n_sample, false);
            if (sh >= 0 && u8_fits(sh)) p = {kPlanU8, sh};
        }
        if (st->bps == 2 && k.n <= kFastMaxFrames && k.n_sample <= kFastMaxSample && k.samp_off) {
            const int sh = fast_sample_shape(k.n, k.n_sample, k.th.absolute != 0);
            if (sh >= 0 && pair_tile_fits(st->dev, st->alloc_bytes, st->bps, st->channels, k, max_pos))
                p = {kPlanFast, sh};
        }
        return p;
    }
    int choice = ctx->choice_for(st->bps, st->channels, k.n, k.th.absolute != 0, sums);
    if (choice < 0) choice = untuned_shape(st->bps, k.n);
    if (choice >= kU8Base) {
        if (u8_fits(choice - kU8Base)) return {kPlanU8, choice - kU8Base};
        // a borrowed stack the wide loads would overrun: the first of the bucket's candidates that
        // stay inside it
        const int b = bucket_for(k.n);
        choice = -1;
        for (int c = 0; b >= 0 && choice < 0 && c < kMaxCand; ++c) {
            const int cand = kBucketCand[st->bps - 1][st->channels >= 3][b][c];
            if (cand >= 0 && (cand < kU8Base || u8_fits(cand - kU8Base))) choice = cand;
        }
        if (choice >= kU8Base) return {kPlanU8, choice - kU8Base};
    }
    if (choice >= 0) {
        if (kShapes[choice].X > 1 && !pair_tile_fits(st->dev, st->alloc_bytes, st->bps, st->channels, k, max_pos))
            choice = st->channels >= 3 ? narrow_shape(choice) : -1;
        if (choice >= 0) p = {kPlanFast, choice};
    }
    return p;
}

int launch_outlier(cp_ctx* ctx, const cp_stack* st, const OutlierK& k, uint64_t max_pos, uint32_t flags,
                   hipStream_t s) {
    const OutlierPlan p = plan_outlier(ctx, st, k, max_pos, flags);
    bool done = false;
    if (p.family == kPlanU8) done = launch_outlier_u8(st->channels, k, p.shape, s);
    else if (p.family == kPlanFast) done = launch_outlier_fast(st->bps, st->channels, k, p.shape, s);
    if (!done) {
        if (st->bps == 1) launch_outlier_generic_b<1>(st, k, s);
        else launch_outlier_generic_b<2>(st, k, s);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(CP_ERR_HIP, "outlier kernel launch: %s", hipGetErrorString(e));
    return CP_OK;
}

template <int B, int C, int PX, bool TABLE>
static void launch_simple_c(const SimpleK& k, bool plain, hipStream_t s) {
    const uint32_t lanes = (k.out_w + PX - 1) / PX;
    dim3 block(256), grid((lanes + 255) / 256, k.out_h);
    if (plain) hipLaunchKernelGGL((simple_plain_kernel<B, C, PX, TABLE>), grid, block, 0, s, k);
    else hipLaunchKernelGGL((simple_kernel<B, C, PX, TABLE>), grid, block, 0, s, k);
}

template <int B, int PX, bool TABLE>
static void launch_simple_b(const cp_stack* st, const SimpleK& k, bool plain, hipStream_t s) {
    switch (st->channels) {
    case 1: launch_simple_c<B, 1, PX, TABLE>(k, plain, s); break;
    case 2: launch_simple_c<B, 2, PX, TABLE>(k, plain, s); break;
    case 3: launch_simple_c<B, 3, PX, TABLE>(k, plain, s); break;
    default: launch_simple_c<B, 4, PX, TABLE>(k, plain, s); break;
    }
}

// Whether a darker/lighter composite with unit weights and no fade takes the whole-number step
// (k_simple.h); one_row: its frames run as one row.  It is the faster one (us, general and whole-number
// step: 64 x 1280x721 RGB8 48 and 28, 300 x 1281x721 RGB8 263 and 148, 200 x 1080p 16-bit mono 166 and
// 148), except that the crops of four 8-bit channels that come from HBM (256 MB and more) suit the
// general step's five waves per SIMD better than eight, unless eight save a round of workgroups: 300 x
// 992x712 (712 groups, one round of either) 182 and 214, 300 x 2592x712 (two of either) 432 and 497,
// but 300 x 1272x712 (two and one) 316 and 249.
static bool whole_numbers(const cp_ctx* ctx, const cp_stack* st, const SimpleK& k, bool one_row) {
    if (st->bps != 1 || st->channels != 4 || one_row) return true;
    const uint64_t blocks = (uint64_t)((k.out_w + 1023u) / 1024u) * k.out_h;
    const uint64_t cus = ctx->cu_count > 0 ? ctx->cu_count : 256;  // a wave per SIMD is a group per CU
    const uint64_t rounds8 = (blocks + 8u * cus - 1) / (8u * cus), rounds5 = (blocks + 5u * cus - 1) / (5u * cus);
    return rounds8 < rounds5 || (uint64_t)k.out_w * k.out_h * 4u * k.n < (256ull << 20);
}

int launch_simple(cp_ctx* ctx, const cp_stack* st, const SimpleK& k_in, hipStream_t s) {
    SimpleK k = k_in;
    bool plain = k.fade.is_none != 0;
    for (uint32_t c = 0; c < st->channels; ++c) plain = plain && k.w[c] == 1.0f;
    // Whole frames are one row: no lane is lost at the row ends, and the waves of a full-HD image
    // fit the device at once (8100 for 8192 slots; row by row 8640, whose last 448 ran alone).  Not in
    // the general step of four 16-bit channels, which is bound by its loads either way (700 x
    // 1280x721 RGBA16 with weights 933 us as one row, 910 us row by row).
    const bool one_row = k.out_w == k.stack_w && (uint64_t)k.out_w * k.out_h < 0x80000000ull &&
                         (plain || st->bps == 1 || st->channels < 4);
    if (one_row) {
        k.out_w *= k.out_h;
        k.out_h = 1;
    }
    plain = plain && whole_numbers(ctx, st, k, one_row);
    // Waves in step (k_simple.h) where one round of them fills three quarters of the device, or half of it
    // on four channels.  us, eight loads in flight and one: RGB8 64 x 1080p (2025 groups for 2048 places)
    // 71.2 and 67.0, 200 x 2592x712 (1802) 198 and 177, but 200 x 1366x768 (1024) 110 and 121 and, in two
    // rounds, 64 x 2048x1080 (2160) 74 and 96; RGBA8 200 x 1366x768 143 and 136, 200 x 1000x667 (651) 95
    // and 115.
    const uint32_t cus = ctx->cu_count > 0 ? (uint32_t)ctx->cu_count : 256u, groups = k.out_w / 1024u;
    k.in_step = one_row && groups >= (st->channels == 4 ? 4u : 6u) * cus && groups < 8u * cus;
    const bool table = k.pos_off.table != nullptr;
    if (st->bps == 1) table ? launch_simple_b<1, 4, true>(st, k, plain, s) : launch_simple_b<1, 4, false>(st, k, plain, s);
    else table ? launch_simple_b<2, 2, true>(st, k, plain, s) : launch_simple_b<2, 2, false>(st, k, plain, s);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(CP_ERR_HIP, "simple kernel launch: %s", hipGetErrorString(e));
    return CP_OK;
}

}  // namespace cp
