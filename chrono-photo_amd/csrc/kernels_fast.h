// kernels_fast.h -- tile shapes of the register-resident outlier kernel and their launch.
//
// A shape (G, F, X) puts G lanes on each group of X pixels and F frames in each lane (G * F >= N);
// a 256-lane workgroup then covers X * 256 / G pixels.  Frame counts fall into buckets; each bucket
// has up to kMaxCand candidate shapes, of this kernel and of the packed-byte one, and the autotuner
// (cp_autotune) measures them on the device and records the fastest per (sample width, channels,
// bucket, threshold kind) in the context.
#pragma once
#include "k_outlier_fast.h"
#include "runtime.h"

namespace cp {

struct TileShape {
    int G, F, X, FS;
};

// Shapes from 10 on put several pixels in each lane (16-bit stacks): one 8- to 16-byte load per
// frame instead of one per pixel, which is what lets a wave's loads reach HBM speed; narrow_shape
// gives the one-pixel shape with the same blocks (3 and 4 channels; for 512 frames one of
// longer blocks).  X is 2
// there, and 4 for one channel (wide_px).  Shapes from 17 on carry an FS-frame block of the
// `--sample` positions.  Before the shapes for 1 and 2 channels, above 512 frames and with a
// sample block, those stacks took the one-lane-per-pixel kernel, which reads every frame from
// L2 once per value bit: 100 x 1937x1091 mono took 4.19 ms and takes 0.176 ms, 300 x 960x541 RGB
// with 48 sample frames 4.41 and 0.380 ms.
constexpr int kNumShapes = 21;
constexpr TileShape kShapes[kNumShapes] = {
    {1, 16, 1, 0}, {1, 32, 1, 0},  {2, 16, 1, 0},  {2, 32, 1, 0},  {4, 16, 1, 0},  {4, 32, 1, 0},  {8, 16, 1, 0},
    {8, 32, 1, 0}, {4, 64, 1, 0},  {8, 64, 1, 0},  {1, 16, 2, 0},  {1, 32, 2, 0},  {2, 32, 2, 0},  {4, 32, 2, 0},
    {8, 32, 2, 0}, {16, 32, 2, 0}, {32, 32, 2, 0}, {4, 32, 2, 16}, {8, 32, 2, 16}, {16, 32, 2, 8}, {32, 32, 2, 4}};
constexpr int kSampleShape0 = 17;
constexpr uint32_t kFastMaxFrames = 32 * 32, kFastMaxSample = 128;
// Pixels per lane of the wide shapes, and of any shape, for a channel count.
constexpr int wide_px(int channels) { return channels == 1 ? 4 : 2; }
constexpr int shape_px(int shape, uint32_t channels) {
    return kShapes[shape].X == 1 ? 1 : wide_px((int)channels);
}
// The smallest 16-bit shape with a sample block that holds n frames and s sample frames, or -1: also
// for short stacks, whose few frames do not pay for the 128-frame groups' pads and search steps (their
// compares and counts are per lane block, not per frame).  There the generic kernel is the faster one
// (us, tile and generic kernel: 5 x 1920x1080 RGB16, all in the sample, rel/2.0/4.0 average 956 and 449,
// 4 frames of RGBA16 1176 and 483 likewise; 20 frames, all in the sample, 1090 and 2876).
// Over 4..24 frames, 3 of them or half or all in the sample, at 641x361 and 1920x1080 with 1-4
// channels, this line costs 0.7 % of the better kernel's time on the geometric mean, 25 % at most (5 x
// 1920x1080 mono, absolute, all in the sample: 176 and 140 us).
inline int fast_sample_shape(uint32_t n, uint32_t s, bool absolute) {
    if (absolute ? n <= 10 && s <= 4 : n + s <= 18) return -1;
    for (int i = kSampleShape0; i < kNumShapes; ++i)
        if ((uint32_t)(kShapes[i].G * kShapes[i].F) >= n && (uint32_t)(kShapes[i].G * kShapes[i].FS) >= s) return i;
    return -1;
}
// Frame-count buckets of the tuned kernel choice.  A choice is a shape of this kernel
// (kShapes index) or, from kU8Base on, a shape of the 8-bit packed-byte kernel (kU8Shapes
// index + kU8Base, kernels_u8.h); each bucket has up to kMaxCand candidates.  kDefault says
// which of them a context takes that was not tuned.
constexpr int kNumBuckets = 9;
constexpr uint32_t kBucketMax[kNumBuckets] = {16, 32, 64, 128, 256, 512, 768, 1024, 1280};
constexpr int kU8Base = 64;
constexpr int kMaxCand = 6;
// [sample bytes - 1][channels >= 3][bucket][candidate]; -1: none
constexpr int kBucketCand[2][2][kNumBuckets][kMaxCand] = {
    // 8-bit, 1-2 channels: the packed-byte kernel only
    {{{kU8Base + 0, kU8Base + 14, -1, -1, -1, -1},
      {kU8Base + 1, kU8Base + 15, -1, -1, -1, -1},
      {kU8Base + 2, kU8Base + 16, kU8Base + 17, kU8Base + 25, -1, -1},
      {kU8Base + 3, kU8Base + 18, -1, -1, -1, -1},
      {kU8Base + 4, kU8Base + 19, -1, -1, -1, -1},
      {kU8Base + 6, kU8Base + 5, kU8Base + 20, -1, -1, -1},
      {kU8Base + 7, kU8Base + 21, -1, -1, -1, -1},
      {kU8Base + 8, kU8Base + 22, -1, -1, -1, -1},
      {kU8Base + 9, kU8Base + 23, -1, -1, -1, -1}},
     // 8-bit, 3-4 channels
     {{0, kU8Base + 0, kU8Base + 14, -1, -1, -1},
      {1, 2, kU8Base + 1, kU8Base + 15, -1, -1},
      {3, 4, kU8Base + 2, kU8Base + 16, kU8Base + 17, kU8Base + 25},
      {5, 6, kU8Base + 3, kU8Base + 18, -1, -1},
      {7, 8, kU8Base + 4, kU8Base + 19, -1, -1},
      {9, kU8Base + 6, kU8Base + 5, kU8Base + 20, -1, -1},
      {kU8Base + 7, kU8Base + 21, -1, -1, -1, -1},
      {kU8Base + 8, kU8Base + 22, -1, -1, -1, -1},
      {kU8Base + 9, kU8Base + 23, -1, -1, -1, -1}}},
    // 16-bit: 1-2 channels and stacks over 512 frames have one shape each (untuned_shape)
    {{{-1, -1, -1, -1, -1, -1}, {-1, -1, -1, -1, -1, -1}, {-1, -1, -1, -1, -1, -1}, {-1, -1, -1, -1, -1, -1},
      {-1, -1, -1, -1, -1, -1}, {-1, -1, -1, -1, -1, -1}, {-1, -1, -1, -1, -1, -1}, {-1, -1, -1, -1, -1, -1},
      {-1, -1, -1, -1, -1, -1}},
     {{10, 0, -1, -1, -1, -1}, {11, 1, -1, -1, -1, -1}, {12, 3, -1, -1, -1, -1}, {13, 5, -1, -1, -1, -1}, {14, 7, -1, -1, -1, -1},
      {15, 9, -1, -1, -1, -1}, {-1, -1, -1, -1, -1, -1}, {-1, -1, -1, -1, -1, -1}, {-1, -1, -1, -1, -1, -1}}}};
// The choice of a context that was not tuned, [sample bytes - 1][channels >= 3][relative][bucket]
// (-1: none): the fastest of the bucket's candidates over 1080p stacks of the scene generator at
// the bucket's limit and at counts inside it, extreme, forward and average modes.  us at 1080p
// RGB, the choice and the first candidate, abs/0.05/0.2 extreme, then rel/2.0/4.0 average:
//   8 bits    16: 40, 49 and 76, 113      32: 68, 81 and 133, 153    64: 132, 180 and 240, 357
//            128: 221, 349 and 502, 661  256: 416, 901 and 988, 1461  512: 852, 2004 and 1910, 2850
//            768: 1190, 1958 and 3002, 6050   1024: 1603, 2401 and 4324, 7801
//   16 bits   16: 108, 121 and 184, 202   64: 233, 268 and 381, 434
//            128: 437 and 740, 904       256: 790 and 1627, 1850
// (two 16-bit pixels per lane load better, one leaves more waves: the three ranks of relative
// thresholds and the few loads of short stacks want the waves).
constexpr int kDefault[2][2][2][kNumBuckets] = {
    {{{kU8Base + 0, kU8Base + 1, kU8Base + 25, kU8Base + 18, kU8Base + 19, kU8Base + 20, kU8Base + 21, kU8Base + 22,
       kU8Base + 23},
      {kU8Base + 14, kU8Base + 15, kU8Base + 25, kU8Base + 18, kU8Base + 19, kU8Base + 20, kU8Base + 21, kU8Base + 22,
       kU8Base + 23}},
     {{kU8Base + 14, kU8Base + 1, kU8Base + 25, kU8Base + 18, kU8Base + 19, kU8Base + 20, kU8Base + 21, kU8Base + 22,
       kU8Base + 23},
      {kU8Base + 14, kU8Base + 15, kU8Base + 25, kU8Base + 18, kU8Base + 19, kU8Base + 20, kU8Base + 21, kU8Base + 22,
       kU8Base + 23}}},
    {{{-1, -1, -1, -1, -1, -1, -1, -1, -1}, {-1, -1, -1, -1, -1, -1, -1, -1, -1}},
     {{0, 1, 3, 13, 14, 15, -1, -1, -1}, {0, 1, 3, 5, 7, 9, -1, -1, -1}}}};
// The same with the mode: sums: an average mode.
inline int default_choice(uint32_t bps, uint32_t channels, int bucket, bool absolute, bool sums) {
    const int c = kDefault[bps - 1][channels >= 3][absolute ? 0 : 1][bucket];
    // 64 frames, the exchange tile and the one whose lanes load their own pixel: four channels
    // fill the exchanged dwords, and one lane's loads are already 4 bytes each (1080p RGBA
    // relative: 286 and 277 us); three channels, relative: 206 and 211 us, but 248 and 240 us in
    // the average modes
    if (c == kU8Base + 25 && (channels == 4 || (channels == 3 && !absolute && sums))) return kU8Base + 17;
    return c;
}

inline int bucket_for(uint32_t n) {
    for (int b = 0; b < kNumBuckets; ++b)
        if (n <= kBucketMax[b]) return b;
    return -1;
}

// The shape of 16-bit stacks whose bucket has no candidates to choose from, or -1: the smallest
// wide one that holds n frames.
inline int untuned_shape(uint32_t bps, uint32_t n) {
    for (int i = 10; bps == 2 && i < kSampleShape0; ++i)
        if ((uint32_t)(kShapes[i].G * kShapes[i].F) >= n) return i;
    return -1;
}

inline int narrow_shape(int shape) {
    for (int i = 0; i < kNumShapes; ++i)
        if (kShapes[i].X == 1 && kShapes[i].G == kShapes[shape].G && kShapes[i].F == kShapes[shape].F) return i;
    return shape == 15 ? 9 : -1;  // 512 frames: 8 lanes of 64
}

template <bool ABS, int B, int C, int G, int F, int X, int FS = 0>
inline void launch_fast_shape(const OutlierK& k, hipStream_t s) {
    constexpr int P = X * 256 / G;
    const uint32_t tiles_x = (k.out_w + P - 1) / P;
    dim3 grid(tiles_x * k.out_h), block(256);
    hipLaunchKernelGGL((outlier_fast_kernel<B, C, G, F, X, FS, ABS>), grid, block, 0, s, k, tiles_x);
}

// ABS: absolute thresholds (k.th.absolute).
template <bool ABS, int B, int C>
inline bool launch_fast_c(const OutlierK& k, int shape, hipStream_t s) {
    if constexpr (C >= 3) {
        switch (shape) {
        case 0: launch_fast_shape<ABS, B, C, 1, 16, 1>(k, s); return true;
        case 1: launch_fast_shape<ABS, B, C, 1, 32, 1>(k, s); return true;
        case 3: launch_fast_shape<ABS, B, C, 2, 32, 1>(k, s); return true;
        case 5: launch_fast_shape<ABS, B, C, 4, 32, 1>(k, s); return true;
        case 7: launch_fast_shape<ABS, B, C, 8, 32, 1>(k, s); return true;
        case 9: launch_fast_shape<ABS, B, C, 8, 64, 1>(k, s); return true;
        default: break;
        }
    }
    if constexpr (B == 1) {
        switch (shape) {
        case 2: launch_fast_shape<ABS, B, C, 2, 16, 1>(k, s); return true;
        case 4: launch_fast_shape<ABS, B, C, 4, 16, 1>(k, s); return true;
        case 6: launch_fast_shape<ABS, B, C, 8, 16, 1>(k, s); return true;
        case 8: launch_fast_shape<ABS, B, C, 4, 64, 1>(k, s); return true;
        default: break;
        }
    } else {
        constexpr int X = wide_px(C);
        switch (shape) {
        case 10: launch_fast_shape<ABS, B, C, 1, 16, X>(k, s); return true;
        case 11: launch_fast_shape<ABS, B, C, 1, 32, X>(k, s); return true;
        case 12: launch_fast_shape<ABS, B, C, 2, 32, X>(k, s); return true;
        case 13: launch_fast_shape<ABS, B, C, 4, 32, X>(k, s); return true;
        case 14: launch_fast_shape<ABS, B, C, 8, 32, X>(k, s); return true;
        case 15: launch_fast_shape<ABS, B, C, 16, 32, X>(k, s); return true;
        case 16: launch_fast_shape<ABS, B, C, 32, 32, X>(k, s); return true;
        case 17: launch_fast_shape<ABS, B, C, 4, 32, X, 16>(k, s); return true;
        case 18: launch_fast_shape<ABS, B, C, 8, 32, X, 16>(k, s); return true;
        case 19: launch_fast_shape<ABS, B, C, 16, 32, X, 8>(k, s); return true;
        case 20: launch_fast_shape<ABS, B, C, 32, 32, X, 4>(k, s); return true;
        default: break;
        }
    }
    return false;
}

// Whether a tile of several pixels per lane may run over this composite: the stack starts on an
// 8-byte boundary (pixels of an even channel count are loaded as they lie, the others realigned
// from dword boundaries), and every read stays inside the stack allocation: the last lane of the
// last row, at the largest frame offset, reads at most 16 bytes from its first sample.
inline bool pair_tile_fits(const void* stack, uint64_t alloc_bytes, uint32_t bps, uint32_t channels,
                           const OutlierK& k, uint64_t max_pos) {
    if ((uintptr_t)stack & 7u) return false;
    const uint64_t X = (uint64_t)wide_px((int)channels), x_last = (k.out_w - 1) / X * X;
    const uint64_t first = max_pos + ((uint64_t)(k.out_h - 1) * k.stack_w + x_last) * channels;
    return first * bps + 16 <= alloc_bytes;
}

// One translation unit per (sample bytes, channels, and for 16 bits threshold kind):
// kernels_fast_b<B>_c<C>[_abs|_rel].hip.
bool launch_fast_b1_c3(const OutlierK& k, int shape, hipStream_t s);
bool launch_fast_b1_c4(const OutlierK& k, int shape, hipStream_t s);
bool launch_fast_b2_c1_abs(const OutlierK& k, int shape, hipStream_t s);
bool launch_fast_b2_c1_rel(const OutlierK& k, int shape, hipStream_t s);
bool launch_fast_b2_c2_abs(const OutlierK& k, int shape, hipStream_t s);
bool launch_fast_b2_c2_rel(const OutlierK& k, int shape, hipStream_t s);
bool launch_fast_b2_c3_abs(const OutlierK& k, int shape, hipStream_t s);
bool launch_fast_b2_c3_rel(const OutlierK& k, int shape, hipStream_t s);
bool launch_fast_b2_c4_abs(const OutlierK& k, int shape, hipStream_t s);
bool launch_fast_b2_c4_rel(const OutlierK& k, int shape, hipStream_t s);

inline bool launch_outlier_fast(uint32_t bps, uint32_t channels, const OutlierK& k, int shape, hipStream_t s) {
    if (bps == 1) {
        if (channels == 3) return launch_fast_b1_c3(k, shape, s);
        return channels == 4 && launch_fast_b1_c4(k, shape, s);
    }
    const bool a = k.th.absolute != 0;
    switch (channels) {
    case 1: return a ? launch_fast_b2_c1_abs(k, shape, s) : launch_fast_b2_c1_rel(k, shape, s);
    case 2: return a ? launch_fast_b2_c2_abs(k, shape, s) : launch_fast_b2_c2_rel(k, shape, s);
    case 3: return a ? launch_fast_b2_c3_abs(k, shape, s) : launch_fast_b2_c3_rel(k, shape, s);
    case 4: return a ? launch_fast_b2_c4_abs(k, shape, s) : launch_fast_b2_c4_rel(k, shape, s);
    default: return false;
    }
}

}  // namespace cp
