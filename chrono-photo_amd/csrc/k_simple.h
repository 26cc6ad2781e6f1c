// k_simple.h -- darker/lighter composite (SimpleProcessor, src/simple.rs:26-176).
//
// Per pixel, frames are visited in index order; value = sum_ch p * w[ch] in channel order
// (f32, no contraction); a strictly smaller (darker) or larger (lighter) value replaces the
// running extreme and blends the frame into the output with fade(t).  The output starts at
// zero and the extreme at +/-f32::MAX (src/simple.rs:77-85).
//
// Streaming kernel: each lane owns PX consecutive output pixels of one row (PX*C*B bytes, a
// multiple of 4 for every channel count with PX = 4 / B), so a wave reads one contiguous
// segment of a frame row; the stack is read exactly once.  A lane's segment is fetched as
// whole aligned dwords: all lanes of a row share the segment's offset within a dword (the row
// start and the frame offset are the only variable parts), so the shift that realigns the
// bytes is wave-uniform.  UF frames are loaded before the first of them is processed,
// keeping UF loads in flight per lane.
//
// With unit weights and no fade (the defaults) a pixel's value is the sum of its samples, a whole
// number that f32 holds exactly, and a new extreme replaces the pixel: PlainPixels keeps the
// pixels packed as they lie in memory and takes one or two dot products, a compare and two
// selects per pixel and frame (simple_plain_kernel).  Bound by HBM.  The general step, about 28 VALU
// instructions per pixel and frame (simple_kernel), is bound by VALU issue: 64 x 1080p RGB8, per call,
// 89.6 us with it and 67.7 us (6.0 TB/s) with whole numbers.
#pragma once
#include "device_common.h"

namespace cp {

// The NB bytes at address a as NB/4 dwords in d[0..NB/4) (d[NB/4] is scratch).  Only dwords
// that hold at least one byte of the segment are read.
template <int B, int NB>
__device__ __forceinline__ void load_segment(const uint8_t* a, uint32_t (&d)[NB / 4 + 1]) {
    const uint32_t s = (uint32_t)(uintptr_t)a & 3u;
    const uint32_t* w = reinterpret_cast<const uint32_t*>(a - s);
    if (s == 0u) {
#pragma unroll
        for (int i = 0; i < NB / 4; ++i) d[i] = w[i];
        d[NB / 4] = 0u;
    } else {
#pragma unroll
        for (int i = 0; i <= NB / 4; ++i) d[i] = w[i];
#pragma unroll
        for (int i = 0; i < NB / 4; ++i) d[i] = __builtin_amdgcn_alignbyte(d[i + 1], d[i], s);
    }
}

template <int B, int C, int PX>
__device__ __forceinline__ void unpack_segment(const uint32_t* d, uint32_t (&in)[PX][4]) {
#pragma unroll
    for (int e = 0; e < PX * C; ++e) {
        const uint32_t word = d[(e * B) / 4];
        const uint32_t sh = 8u * (uint32_t)((e * B) % 4);
        in[e / C][e % C] = B == 1 ? (word >> sh) & 0xFFu : (word >> sh) & 0xFFFFu;
    }
}

template <int B, int C, int PX>
__device__ __forceinline__ void simple_step(const SimpleK& k, bool darker, int32_t t, int32_t N,
                                            const uint32_t (&in)[PX][4], float (&ext)[PX], uint32_t (&out)[PX][4]) {
    constexpr uint32_t maxv = B == 1 ? 255u : 65535u;
    bool have_fade = false;  // fade(t) computed lazily, once per frame
    float fade = 1.0f;
#pragma unroll
    for (int p = 0; p < PX; ++p) {
        float value = 0.0f;
#pragma unroll
        for (int ch = 0; ch < C; ++ch) value += (float)in[p][ch] * k.w[ch];
        const bool is_ext = darker ? (value < ext[p]) : (value > ext[p]);
        if (is_ext) {
            ext[p] = value;
            if (!have_fade) { fade = fade_pick(k.fade, t, N, k.frame_offset); have_fade = true; }
            const float f = fade;
            if (f > 0.0f) {
                if (f >= 1.0f) {
#pragma unroll
                    for (int ch = 0; ch < C; ++ch) out[p][ch] = in[p][ch];
                } else {
#pragma unroll
                    for (int ch = 0; ch < C; ++ch) {
                        const float aa = (float)out[p][ch];
                        out[p][ch] = sat_cast(roundf(aa + ((float)in[p][ch] - aa) * f), maxv);
                    }
                }
            }
        }
    }
}

// The running extremes of a lane's PX pixels for unit weights without fade.  d: the segment's
// dwords.  Pixel p's samples start at bit p * C * 8 * B of the segment.
template <int B, int C, int PX>
struct PlainPixels {
    static constexpr int ND = PX * C * B / 4;
    static constexpr int BITS = C * 8 * B;  // per pixel
    uint32_t ext[PX];
    uint32_t out[ND];
    __device__ __forceinline__ void init() {
#pragma unroll
        for (int p = 0; p < PX; ++p) ext[p] = 0xFFFFFFFFu;  // above every key but a black pixel's, and out is black
#pragma unroll
        for (int i = 0; i < ND; ++i) out[i] = 0u;
    }
    // Bits of dword i that belong to pixel p.
    static constexpr uint32_t mask(int i, int p) {
        uint32_t m = 0;
        for (int b = 0; b < 32; ++b)
            if ((32 * i + b) / BITS == p) m |= 1u << b;
        return m;
    }
    __device__ __forceinline__ void step(const uint32_t* d, bool darker) {
        bool take[PX];
#pragma unroll
        for (int p = 0; p < PX; ++p) {
            uint32_t v = 0;
#pragma unroll
            for (int i = 0; i < ND; ++i) {
                const uint32_t m = mask(i, p);
                if (m == 0) continue;
                if constexpr (B == 1) v = __builtin_amdgcn_udot4(d[i], m & 0x01010101u, v, false);
                else v = __builtin_amdgcn_udot2(__builtin_bit_cast(us2s, d[i]), __builtin_bit_cast(us2s, m & 0x00010001u), v, false);
            }
            // the lighter mode compares -v - 1 with the same order; v < 2^18
            const uint32_t key = darker ? v : ~v;
            take[p] = key < ext[p];
            ext[p] = take[p] ? key : ext[p];
        }
#pragma unroll
        for (int i = 0; i < ND; ++i) {
            uint32_t o = out[i];
#pragma unroll
            for (int p = 0; p < PX; ++p) {
                const uint32_t m = mask(i, p);
                if (m == 0) continue;
                if (m == 0xFFFFFFFFu) o = take[p] ? d[i] : o;
                else o = (o & ~m) | ((take[p] ? d[i] : o) & m);
            }
            out[i] = o;
        }
    }
    typedef unsigned short us2s __attribute__((ext_vector_type(2)));
};

// PLAIN: unit weights and no fade.  TABLE: the frame positions' offsets come from a table (crops,
// uneven selections) or from their spacing; a test of that per frame waited for each entry before
// it asked for the next (20 x 1280x721 mono lighter with weights and crops 23.3 us, 22.4 us without
// it; 700 x 16 bits, two channels, 512 and 453 us with the register bound below gone as well).
template <int B, int C, int PX, bool PLAIN, bool TABLE>
__device__ __forceinline__ void simple_pixels(const SimpleK& k) {
    uint32_t x0 = (blockIdx.x * blockDim.x + threadIdx.x) * PX;
    const uint32_t y = blockIdx.y;
    if (x0 >= k.out_w || y >= k.out_h) return;
    // A row that ends inside a lane's pixels: the lanes of its last wave all step back to end with
    // it, so that every lane holds whole segments and the wave keeps one shift.  The pixels that
    // lane 0 then shares with the wave before are that wave's to store.  Only a row of a single
    // wave keeps a partial lane, which loads one frame's samples after another's (a latency
    // each: 48 x 1281x721 RGB8 took 43.6 us with one at the end of the frame and takes 23.5 us so,
    // 300 frames 315 and 148 us; the same at 1280x721 22.8 and 152 us).
    const uint32_t part = k.out_w % PX;
    const uint32_t wave_x0 = __builtin_amdgcn_readfirstlane((blockIdx.x * 256u + (threadIdx.x & ~63u)) * PX);
    const bool back = part != 0u && wave_x0 != 0u && k.out_w - wave_x0 <= 64u * PX;
    if (back) x0 -= PX - part;
    const uint32_t npx = min((uint32_t)PX, k.out_w - x0);
    const bool darker = k.darker != 0;
    float ext[PX];
    uint32_t out[PX][4];
#pragma unroll
    for (int p = 0; p < PX; ++p) {
        ext[p] = darker ? 3.40282347e+38f : -3.40282347e+38f;
#pragma unroll
        for (int ch = 0; ch < 4; ++ch) out[p][ch] = 0;
    }
    const uint64_t pix = ((uint64_t)y * k.stack_w + x0) * C;
    const int32_t N = (int32_t)k.n;
    constexpr int NB = PX * C * B;
    constexpr bool WHOLE = NB % 4 == 0;
    if constexpr (PLAIN && WHOLE) {
        if (npx == (uint32_t)PX) {
            constexpr int UF = 8, ND = NB / 4;  // UF frames in flight
            typedef uint32_t words __attribute__((ext_vector_type(ND), aligned(4)));
            typedef uint32_t words1 __attribute__((ext_vector_type(ND + 1), aligned(4)));
            const uintptr_t base = (uintptr_t)k.stack + pix * B;
            const uint32_t base_sh = __builtin_amdgcn_readfirstlane((uint32_t)base & 3u);  // of the whole row
            PlainPixels<B, C, PX> px;
            px.init();
            uint32_t d[UF][ND + 1], sh[UF];
            auto load = [&](int u, uint64_t off) {
                // whole dwords from the one that holds the first byte to the one that holds the
                // last; the lanes of a wave share the shift.  The last dword of a shifted segment
                // comes with the others in the crops of 8-bit stacks (200 x 1926x1086 RGB8 333 us
                // with a load of its own, 303 us so), and by itself elsewhere: whole images seldom
                // shift, and the wider loads are slower even where they do not run (64 x 1280x721
                // mono 19.7 us with them, 16.2 us without), crops of 16 bits 200 x 1926x1086 mono
                // 192 and 163 us.
                constexpr bool TOGETHER = B == 1 && TABLE && ND < 4;
                const uintptr_t a = base + off * B;
                sh[u] = (base_sh + (uint32_t)off * B) & 3u;
                const uintptr_t w = a & ~(uintptr_t)3;
                if (TOGETHER && sh[u] != 0u) {
                    const words1 v = *(const __attribute__((address_space(1))) words1*)w;
#pragma unroll
                    for (int i = 0; i <= ND; ++i) d[u][i] = v[i];
                    return;
                }
                const words v = *(const __attribute__((address_space(1))) words*)w;
#pragma unroll
                for (int i = 0; i < ND; ++i) d[u][i] = v[i];
                d[u][ND] = 0u;
                if (!TOGETHER && sh[u] != 0u) d[u][ND] = *(const __attribute__((address_space(1))) uint32_t*)(w + NB);
            };
            int32_t t = 0;
            for (; t + UF <= N; t += UF) {
#pragma unroll
                for (int u = 0; u < UF; ++u) {
                    load(u, k.pos_off.wave_at<TABLE>(t + u));
                    // Where the waves fill the device, one wide load in flight in each is enough, and
                    // waves that wait for it stay on the same frame, whose rows follow one another
                    // in memory (64 x 1080p RGB8 lighter 71.2 us with eight in flight, 67.0 us so).
                    if (B == 1 && C >= 3 && !TABLE && k.in_step) __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
                }
#pragma unroll
                for (int u = 0; u < UF; ++u) {
                    uint32_t w[ND];
#pragma unroll
                    for (int i = 0; i < ND; ++i) w[i] = __builtin_amdgcn_alignbyte(d[u][i + 1], d[u][i], sh[u]);
                    px.step(w, darker);
                }
            }
            for (; t < N; ++t) {
                load(0, k.pos_off.wave_at<TABLE>(t));
                uint32_t w[ND];
#pragma unroll
                for (int i = 0; i < ND; ++i) w[i] = __builtin_amdgcn_alignbyte(d[0][i + 1], d[0][i], sh[0]);
                px.step(w, darker);
            }
            const uint64_t at = ((uint64_t)y * k.out_w + x0) * C;
            const uint32_t skip = back && __lane_id() == 0u ? PX - part : 0u;
            if (skip != 0u) {
                uint32_t v[PX][4];
                unpack_segment<B, C, PX>(px.out, v);
#pragma unroll
                for (int e = 0; e < PX * C; ++e)
                    if ((uint32_t)(e / C) >= skip) store_sample<B>(k.out_px, at + e, v[e / C][e % C]);
                return;
            }
            typedef uint32_t out_words __attribute__((ext_vector_type(ND), aligned(B)));
            out_words o;
#pragma unroll
            for (int i = 0; i < ND; ++i) o[i] = px.out[i];
            *(__attribute__((address_space(1))) out_words*)((uintptr_t)k.out_px + at * B) = o;
            return;
        }
    }
    if (WHOLE && npx == (uint32_t)PX) {
        constexpr int UF = 8;
        int32_t t = 0;
        for (; t + UF <= N; t += UF) {
            uint32_t d[UF][NB / 4 + 1];
#pragma unroll
            for (int u = 0; u < UF; ++u) load_segment<B, NB>(k.stack + (k.pos_off.wave_at<TABLE>(t + u) + pix) * B, d[u]);
#pragma unroll
            for (int u = 0; u < UF; ++u) {
                uint32_t in[PX][4];
                unpack_segment<B, C, PX>(d[u], in);
                simple_step<B, C, PX>(k, darker, t + u, N, in, ext, out);
            }
        }
        for (; t < N; ++t) {
            uint32_t d[NB / 4 + 1];
            load_segment<B, NB>(k.stack + (k.pos_off.wave_at<TABLE>(t) + pix) * B, d);
            uint32_t in[PX][4];
            unpack_segment<B, C, PX>(d, in);
            simple_step<B, C, PX>(k, darker, t, N, in, ext, out);
        }
    } else {
        for (int32_t t = 0; t < N; ++t) {
            const uint64_t base = k.pos_off.wave_at<TABLE>(t) + pix;
            uint32_t in[PX][4];
#pragma unroll
            for (int e = 0; e < PX * C; ++e)
                in[e / C][e % C] = (uint32_t)(e / C) < npx ? load_sample<B>(k.stack, base + e) : 0u;
            simple_step<B, C, PX>(k, darker, t, N, in, ext, out);
        }
    }
    const uint32_t skip = back && __lane_id() == 0u ? PX - part : 0u;
    const uint64_t o = ((uint64_t)y * k.out_w + x0) * C;
#pragma unroll
    for (int p = 0; p < PX; ++p) {
        if ((uint32_t)p >= npx) break;
        if ((uint32_t)p < skip) continue;
#pragma unroll
        for (int ch = 0; ch < C; ++ch) store_sample<B>(k.out_px, o + p * C + ch, out[p][ch]);
    }
}

// The general step takes the registers it needs (22 to 82); held to the 64 of eight waves per SIMD,
// four 16-bit channels spilled (64 x 1280x721 RGBA16 lighter with weights and crops 99.9 us, 95.9 us
// without the bound; 90 x RGBA8 139 and 118 us).  The whole-number step fits eight waves.
template <int B, int C, int PX, bool TABLE>
__global__ void __launch_bounds__(256) simple_kernel(SimpleK k) {
    simple_pixels<B, C, PX, false, TABLE>(k);
}

template <int B, int C, int PX, bool TABLE>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) simple_plain_kernel(SimpleK k) {
    simple_pixels<B, C, PX, true, TABLE>(k);
}

}  // namespace cp
