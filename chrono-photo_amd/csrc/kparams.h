// kparams.h -- kernel argument blocks (plain data, shared by host and device code).
#pragma once
#include <stdint.h>

namespace cp {

struct ThresholdK {
    int32_t absolute;
    float min, max, scale;
};

struct FadeK {
    int32_t is_none, repeat, absolute, offset;
    uint32_t len;
    const float* values;  // device table
};

// Per-pixel diagnostics; layout shared with the C ABI (cp_pixel_stats).
struct PixelStats {
    float median[4];
    float iqr_inv[4];
    uint32_t num_outliers;
    uint32_t max_index;
    float max_dist_sq;
    uint32_t bg_index;
    uint32_t warning;
    uint32_t pad;
};

// Element offsets of a composite's frame positions: a device table, or without one an even
// spacing.  Whole stacks, video windows and frame ranges are evenly spaced, and their calls need
// no copy of a table in front of the kernel.
struct PosK {
    const uint64_t* table;  // n offsets, or null
    uint64_t first;
    int64_t step;
    __device__ __forceinline__ uint64_t operator[](uint32_t t) const {
        return table ? table[t] : first + (uint64_t)(step * (int64_t)t);
    }
    // The same for a kernel that knows at compile time which of the two it was given.
    template <bool TABLE>
    __device__ __forceinline__ uint64_t at(uint32_t t) const {
        return TABLE ? table[t] : first + (uint64_t)(step * (int64_t)t);
    }
    // at() for a position that a wave's lanes share.  The offset stays scalar: left to itself the
    // compiler turns the spacing into a pointer per lane and frame in flight (80 vector registers
    // instead of 64 in the widest darker/lighter kernel).
    template <bool TABLE>
    __device__ __forceinline__ uint64_t wave_at(uint32_t t) const {
        const uint64_t o = at<TABLE>(t);
        return (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(o >> 32)) << 32 |
               (uint32_t)__builtin_amdgcn_readfirstlane((int)o);
    }
};

// One composite over a device-resident stack.  Frame position t (0..n-1) reads sample
// (x, y, ch) at element index pos_off[t] + (y * stack_w + x) * C + ch, where pos_off folds
// the stack slot and the per-frame crop origin.
struct OutlierK {
    const uint8_t* stack;
    PosK pos_off;                // n element offsets
    const uint32_t* sample_mask; // bit t set: position t is in the median sample (null: all)
    const uint64_t* samp_off;    // element offsets of the n_sample sample positions (null: all)
    uint32_t n, n_sample;
    uint32_t stack_w;            // row pitch in pixels
    uint32_t out_w, out_h;
    int32_t frame_offset;
    ThresholdK th;
    int32_t background, outlier;
    float w[4];
    FadeK fade;
    uint64_t seed;
    uint64_t pix_base;           // image index of output pixel (0, 0): row bands draw the same random numbers
    void* out_px;
    uint8_t* out_mask;
    unsigned long long* warnings;
    PixelStats* stats;
};

struct SimpleK {
    const uint8_t* stack;
    PosK pos_off;
    uint32_t n;
    uint32_t stack_w;
    uint32_t out_w, out_h;
    int32_t frame_offset;
    int32_t darker;
    uint32_t in_step;  // whole-number step: one load at a time per wave (set by the launch)
    float w[4];
    FadeK fade;
    void* out_px;
};

}  // namespace cp
