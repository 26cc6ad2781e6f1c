// k_shake.h -- camera-shake offsets (ShakeAnalyzer, src/shake.rs:190-385).
//
// For every frame f >= 1 and every candidate offset (ox, oy) in [-s, s]^2 the kernel sums
// (win - img)^2 over all anchors, window pixels (2r+1)^2 and channels, where win is the
// anchor window of frame 0 (fill_windows, :315-343) and img the frame-f pixel displaced by
// (ox, oy) (calc_diffs, :345-385).  The offset with the smallest sum wins; ties go to the
// first index in row-major (oy, ox) order (min_by_key, :294-297).
//
// u8 sums wrap in i32 like the reference (release build, overflow-checks = false): the
// kernels sum exactly and the arg-min reads each total modulo 2^32, which is that wrapped
// value.  u16 sums are exact 64-bit integers.
//
// The sums on the matrix cores.  A difference does not change when a constant is taken from
// both samples, so the samples are centred: 8-bit ones become v - 128, 16-bit ones
// v - 128 * 257 = 256 h + l, with h and l signed bytes (the sample's two bytes less 128).
// Each candidate's sum is
//   sum (w - v)^2 = sum w^2 + sum v^2 - 2 sum w*v,
// and for one window row dy the last term is a product of matrices: with the samples q of a
// region row as the contraction index, A[ox][q] = w[dy][q - ox * C] (zero outside the window
// row; the same row at another byte offset for every ox) times B[q][oy] = v[oy + dy][q].
// Signed-byte MFMA (16x16x64) accumulates it over q and dy in exact 32-bit sums: one product
// per slab of 64 samples for 8-bit frames, and h*h, h*l + l*h and l*l for 16-bit ones.
//
// Work split.  A workgroup owns one (frame, anchor, block of up to 32 x 32 candidates, chunk
// of window rows) and stages the chunk's window rows and the region rows they reach in LDS as
// byte planes.  Its four waves take every fourth window row; each wave keeps all 2 x 2 tiles
// of its candidate block, so that a slab costs 8 LDS reads for 16 MFMAs (waves that each took
// one tile would read twice as much).  The window rows carry zeros on both sides; a lane reads
// its 16 bytes at any byte offset from the dword at or below them and realigns them.
// sum v^2 comes from per-row box sums by signed dot products, sum w^2 is one constant per
// analysis (the frame-1 workgroups add it to a spare slot of the table; the arg-min kernel adds
// it back).  The waves' sums meet in LDS (64-bit integer adds, any order) and one atomic per
// candidate adds the workgroup's part to the frame's table.
//
// 256 x 4K RGB16, 5 anchors, r = 32, s = 12, per call: 0.78 ms with f64 products on the vector
// units (bound by their issue), 0.206 ms with the matrix cores (0.245 ms before the staging loads
// were all in flight at once and the box sums of a candidate were added up once).  Staging, box
// sums and products follow one another in a workgroup; three workgroups per CU overlap them.
#pragma once
#include "device_common.h"

namespace cp {

struct ShakeK {
    const uint8_t* stack;
    const uint64_t* pos_off;  // element offset of each frame position (no crop)
    uint32_t stack_w;
    uint32_t n;
    const int32_t* anchors;   // device, 2 per anchor
    uint32_t n_anchors;
    int32_t r, s;
    int32_t chunk_rows;       // window rows per workgroup
    int32_t n_chunks;         // ceil((2r+1) / chunk_rows)
    int32_t cand_rows;        // candidate rows oy per workgroup (at most 32)
    int32_t cand_chunks;      // ceil((2s+1) / cand_rows)
    int32_t cand_cols;        // candidate columns ox per workgroup (at most 32)
    int32_t col_chunks;       // ceil((2s+1) / cand_cols)
    uint32_t group0;          // first (chunk, candidate block, anchor) combination of this launch
    unsigned long long* sums; // [n][(2s+1)^2], then the sum of squared window samples
    int32_t* offsets;         // [n][2]
};

// LDS layout of one workgroup for `rows` window rows and a block of orows x ocols candidates:
// region byte planes (rows + orows - 1 rows of rpitch bytes each), window byte planes (rows
// rows of wpitch bytes; the window row starts at byte wlead), box sums (i64, one per region row
// and candidate column) and the block's totals (i64).
struct ShakeLds {
    uint32_t rlen;    // samples of a region row that the block reaches
    uint32_t slabs;   // slabs of 64 samples
    uint32_t rpitch, wpitch, wlead;
    uint32_t srows;
    uint64_t win_off, rq_off, tot_off, bytes;
};
__host__ __device__ inline ShakeLds shake_lds(int32_t rows, int32_t orows, int32_t ocols, int32_t r, int32_t channels,
                                             int32_t planes) {
    ShakeLds l;
    const uint32_t otile = ocols > 16 ? 32u : 16u;  // columns covered by the tiles
    l.srows = (uint32_t)(rows + orows - 1);
    l.rlen = (uint32_t)((2 * r + 1 + ocols - 1) * channels);
    l.slabs = (l.rlen + 63u) / 64u;
    l.rpitch = l.slabs * 64u + 16u;  // rows 16 bytes apart modulo 64: their reads spread over the banks
    l.wlead = (otile * (uint32_t)channels + 15u) / 16u * 16u;
    l.wpitch = l.wlead + l.slabs * 64u + 16u;
    l.win_off = (uint64_t)l.srows * l.rpitch * planes;
    l.rq_off = l.win_off + (uint64_t)rows * l.wpitch * planes;
    l.tot_off = l.rq_off + (uint64_t)l.srows * ocols * 8u;
    l.bytes = l.tot_off + (uint64_t)orows * ocols * 8u;
    return l;
}

typedef int i32x4 __attribute__((ext_vector_type(4)));

// Eight samples from element e of a row that holds `len` >= 8 or fewer samples, centred, as bytes
// (hi and lo planes for 16-bit samples, lo alone for 8-bit ones); samples past len are zero.  A row
// of eight samples or more is read without a branch: where the eight would pass its end, the
// row's last eight are read and shifted.
template <int B>
__device__ __forceinline__ void load_centred8(const uint8_t* row, uint32_t e, uint32_t len, uint2& hi, uint2& lo) {
    typedef uint32_t words __attribute__((ext_vector_type(2 * B), aligned(B)));
    typedef const __attribute__((address_space(1))) words gwords;
    const uint32_t at = min(e, len >= 8u ? len - 8u : 0u), past = min(e - at, 8u);  // samples to shift out
    uint32_t w[2 * B];
    if (len >= 8u) {  // the same for every lane
        const words v = *(gwords*)(uintptr_t)(row + at * B);
#pragma unroll
        for (int i = 0; i < 2 * B; ++i) w[i] = v[i];
    } else {
#pragma unroll
        for (int i = 0; i < 2 * B; ++i) w[i] = 0x80808080u;
#pragma unroll
        for (uint32_t i = 0; i < 8u; ++i) {
            if (i >= len) break;
            const uint32_t bit = 8u * B * i, v = load_sample<B>(row, i);
            w[bit / 32u] = (w[bit / 32u] & ~((B == 1 ? 0xFFu : 0xFFFFu) << (bit % 32u))) | (v << (bit % 32u));
        }
    }
    auto shifted = [&](uint32_t a, uint32_t b) {  // the plane's eight bytes less `past`, zeros behind
        const uint64_t v = (((uint64_t)(b ^ 0x80808080u) << 32) | (a ^ 0x80808080u));
        const uint64_t r = past >= 8u ? 0ull : v >> (8u * past);
        return uint2{(uint32_t)r, (uint32_t)(r >> 32)};
    };
    if constexpr (B == 1) {
        lo = shifted(w[0], w[1]);
        hi = uint2{0u, 0u};
    } else {
        lo = shifted(__builtin_amdgcn_perm(w[1], w[0], 0x06040200u),
                     __builtin_amdgcn_perm(w[2 * B - 1], w[2 * B - 2], 0x06040200u));
        hi = shifted(__builtin_amdgcn_perm(w[1], w[0], 0x07050301u),
                     __builtin_amdgcn_perm(w[2 * B - 1], w[2 * B - 2], 0x07050301u));
    }
}

// Stages `rows` rows of `len` samples (row y at base + y * stride bytes) as byte planes: plane p
// of row y at dst + (p * rows + y) * pitch; samples past len are zero.  groups: eights of bytes
// per row.  Sixteen lanes share a row, so that no lane divides and a row's loads are contiguous;
// the loads of R rows are all in flight before the first is used.
template <int B, int R>
__device__ __forceinline__ void stage_rows(const uint8_t* base, uint64_t stride, uint32_t rows, uint32_t len,
                                           uint32_t groups, uint8_t* dst, uint32_t pitch) {
    constexpr uint32_t U = 3;  // groups of a row per lane and round
    const uint32_t gx = threadIdx.x & 15u, y0 = threadIdx.x >> 4;
    for (uint32_t yb = 0; yb < rows; yb += 16u * R) {
        for (uint32_t qb = 0; qb < groups; qb += 16u * U) {
            uint2 hi[R][U], lo[R][U];
#pragma unroll
            for (uint32_t r = 0; r < R; ++r) {
                const uint32_t y = min(yb + 16u * r + y0, rows - 1u);
#pragma unroll
                for (uint32_t u = 0; u < U; ++u)
                    load_centred8<B>(base + y * stride, min(qb + 16u * u + gx, groups - 1u) * 8u, len, hi[r][u], lo[r][u]);
            }
#pragma unroll
            for (uint32_t r = 0; r < R; ++r) {
                const uint32_t y = yb + 16u * r + y0;
#pragma unroll
                for (uint32_t u = 0; u < U; ++u) {
                    const uint32_t q = qb + 16u * u + gx;
                    if (y >= rows || q >= groups) continue;
                    *reinterpret_cast<uint2*>(dst + y * pitch + q * 8u) = lo[r][u];
                    if constexpr (B == 2) *reinterpret_cast<uint2*>(dst + (rows + y) * pitch + q * 8u) = hi[r][u];
                }
            }
        }
    }
}

// Sum of squares of the packed centred samples of one dword (and its high plane's).
template <int B>
__device__ __forceinline__ void square_acc(uint32_t hi, uint32_t lo, int32_t& hh, int32_t& hl, int32_t& ll) {
    ll = __builtin_amdgcn_sdot4((int)lo, (int)lo, ll, false);
    if constexpr (B == 2) {
        hl = __builtin_amdgcn_sdot4((int)hi, (int)lo, hl, false);
        hh = __builtin_amdgcn_sdot4((int)hi, (int)hi, hh, false);
    }
}

// 65536 hh + 512 hl + ll: the squares' sum of samples 256 h + l (hl once per sample).
template <int B>
__device__ __forceinline__ long long square_total(int32_t hh, int32_t hl, int32_t ll) {
    if constexpr (B == 1) return ll;
    else return ((long long)hh << 16) + ((long long)hl << 9) + ll;
}

// Sum over the eight adjacent lanes of a half-row (xor 1, xor 2, half-row mirror).
__device__ __forceinline__ int32_t grp8_sum(int32_t v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x141, 0xF, 0xF, true);
    return v;
}

template <int B, int C>
__global__ void __launch_bounds__(256) shake_ssd_kernel(ShakeK k) {
    constexpr int PL = B;  // byte planes: low, then high
    extern __shared__ __align__(16) uint8_t lds[];
    const uint32_t f = blockIdx.x + 1;
    // (chunk of window rows, block of candidate columns, block of candidate rows, anchor)
    uint32_t q = k.group0 + blockIdx.y;
    const int32_t zc = (int32_t)(q % (uint32_t)k.n_chunks);
    q /= (uint32_t)k.n_chunks;
    const int32_t xc = (int32_t)(q % (uint32_t)k.col_chunks);
    q /= (uint32_t)k.col_chunks;
    const int32_t yc = (int32_t)(q % (uint32_t)k.cand_chunks);
    const uint32_t a = q / (uint32_t)k.cand_chunks;
    const int32_t r = k.r, s = k.s;
    const int32_t size = 2 * r + 1, ssize = 2 * s + 1;
    const int32_t c0 = zc * k.chunk_rows, crows = min(size, c0 + k.chunk_rows) - c0;
    const int32_t oy0 = yc * k.cand_rows, orows = min(ssize, oy0 + k.cand_rows) - oy0;
    const int32_t ox0 = xc * k.cand_cols, ocols = min(ssize, ox0 + k.cand_cols) - ox0;
    const ShakeLds lay = shake_lds(crows, orows, ocols, r, C, PL);
    uint8_t* region = lds;
    uint8_t* win = lds + lay.win_off;
    long long* rq = reinterpret_cast<long long*>(lds + lay.rq_off);
    unsigned long long* tot = reinterpret_cast<unsigned long long*>(lds + lay.tot_off);
    const uint32_t tid = threadIdx.x;
    const int32_t cx = k.anchors[2 * a], cy = k.anchors[2 * a + 1];
    const uint32_t srows = lay.srows, wsamples = (uint32_t)(size * C);

    // ---- stage: region rows oy0 + c0 .. of frame f, window rows c0 .. of frame 0 with zeros
    // around them
    {
        const uint64_t stride = (uint64_t)k.stack_w * C * B;
        const uint8_t* rbase =
            k.stack + (k.pos_off[f] + ((uint64_t)(cy - s - r + oy0 + c0) * k.stack_w + (cx - s - r + ox0)) * C) * B;
        stage_rows<B, 3>(rbase, stride, srows, lay.rlen, lay.slabs * 8u, region, lay.rpitch);
        const uint8_t* wbase = k.stack + (k.pos_off[0] + ((uint64_t)(cy - r + c0) * k.stack_w + (cx - r)) * C) * B;
        stage_rows<B, 1>(wbase, stride, (uint32_t)crows, wsamples, (lay.wpitch - lay.wlead) / 8u, win + lay.wlead,
                      lay.wpitch);
        const uint32_t lead = lay.wlead / 4u, wrows = (uint32_t)crows * PL;
        for (uint32_t i = tid; i < wrows * lead; i += 256u)
            *reinterpret_cast<uint32_t*>(win + (i / lead) * lay.wpitch + (i % lead) * 4u) = 0u;
    }
    __syncthreads();

    // ---- sum w^2, once per (anchor, window chunk): the same for every frame and candidate
    if (f == 1 && xc == 0 && yc == 0) {
        const uint32_t words = (wsamples + 3u) / 4u;
        unsigned long long w2 = 0;
        for (uint32_t i = tid; i < (uint32_t)crows * words; i += 256u) {
            const uint32_t y = i / words, e = lay.wlead + (i - y * words) * 4u;
            const uint32_t lo = *reinterpret_cast<const uint32_t*>(win + y * lay.wpitch + e);
            uint32_t hi = 0;
            if constexpr (B == 2) hi = *reinterpret_cast<const uint32_t*>(win + ((uint32_t)crows + y) * lay.wpitch + e);
            int32_t hh = 0, hl = 0, ll = 0;
            square_acc<B>(hi, lo, hh, hl, ll);
            w2 += (unsigned long long)square_total<B>(hh, hl, ll);
        }
        if (w2 != 0) atomicAdd(k.sums + (uint64_t)k.n * ssize * ssize, w2);
    }

    // ---- rq[y][x] = squares' sum over the window width from candidate column x.  Per row, lane i
    // of eight sums every eighth dword of the first window, the eight meet by DPP, and lane i
    // then goes on from the sum of what enters and leaves on the way to its own columns.
    {
        constexpr uint32_t PITCH8 = 8u;
        const uint32_t sub = tid & (PITCH8 - 1u);
        const uint32_t per = ((uint32_t)ocols + PITCH8 - 1u) / PITCH8;  // columns per lane
        const uint32_t words = wsamples / 4u;
        for (uint32_t y0 = 0; y0 < srows; y0 += 256u / PITCH8) {
            const uint32_t yr = y0 + tid / PITCH8, y = min(yr, srows - 1u);
            const uint8_t* plo = region + y * lay.rpitch;
            const uint8_t* phi = region + (srows + y) * lay.rpitch;
            int32_t hh = 0, hl = 0, ll = 0;
            auto one = [&](uint32_t at, int32_t sign) {
                const int32_t l = (int8_t)plo[at];
                ll += sign * l * l;
                if constexpr (B == 2) {
                    const int32_t h = (int8_t)phi[at];
                    hl += sign * h * l;
                    hh += sign * h * h;
                }
            };
#pragma unroll 4
            for (uint32_t b = sub; b < words; b += PITCH8) {
                uint32_t hi = 0;
                if constexpr (B == 2) hi = *reinterpret_cast<const uint32_t*>(phi + 4u * b);
                square_acc<B>(hi, *reinterpret_cast<const uint32_t*>(plo + 4u * b), hh, hl, ll);
            }
            if (sub < wsamples % 4u) one(words * 4u + sub, 1);
            ll = grp8_sum(ll);
            if constexpr (B == 2) {
                hl = grp8_sum(hl);
                hh = grp8_sum(hh);
            }
            // the step from column x to x + 1 takes pixel x out and pixel x + size in: lanes step
            // over their own columns, then take the steps of the lanes before them
            const long long first = square_total<B>(hh, hl, ll);
            hh = hl = ll = 0;
            const uint32_t xa = min(sub * per, (uint32_t)ocols), xb = min(xa + per, (uint32_t)ocols);
            for (uint32_t x = xa; x < xb; ++x) {
                if (yr < srows) rq[y * (uint32_t)ocols + x] = square_total<B>(hh, hl, ll);
                if (x + 1u < (uint32_t)ocols) {
#pragma unroll
                    for (uint32_t c = 0; c < (uint32_t)C; ++c) {
                        one(x * C + c, -1);
                        one(x * C + wsamples + c, 1);
                    }
                }
            }
            long long before = first, step = square_total<B>(hh, hl, ll);
#pragma unroll
            for (uint32_t j = 0; j < PITCH8 - 1u; ++j) {
                const long long v = __shfl(step, (int)((tid & 56u) + j));
                before += j < sub ? v : 0;
            }
            if (yr < srows)
                for (uint32_t x = xa; x < xb; ++x) rq[y * (uint32_t)ocols + x] += before;
        }
    }

    // ---- sum w * v by MFMA: tile rows are candidate columns ox, tile columns candidate rows oy
    const uint32_t lane = tid & 63u, wave = tid >> 6, m16 = lane & 15u, kq = lane >> 4;
    i32x4 acc[2][2][B == 2 ? 3 : 1];  // [ox tile][oy tile][l*l (, h*l + l*h, h*h)]
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int p = 0; p < (B == 2 ? 3 : 1); ++p) acc[i][j][p] = i32x4{0, 0, 0, 0};
    const bool ox2 = ocols > 16, oy2 = orows > 16;
    // byte of the window row that meets region sample 0 in this lane's candidate column
    uint32_t wal[2], wsh[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const uint32_t at = lay.wlead + kq * 16u - min(m16 + 16u * i, ox2 ? 31u : 15u) * C;
        wal[i] = at & ~3u;
        wsh[i] = at & 3u;
    }
    uint32_t brow[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) brow[j] = min(m16 + 16u * j, (uint32_t)orows - 1u) * lay.rpitch + kq * 16u;
    for (uint32_t dy = wave; dy < (uint32_t)crows; dy += 4u) {
        const uint8_t* wr = win + dy * lay.wpitch;
        const uint8_t* rr = region + dy * lay.rpitch;
        for (uint32_t sl = 0; sl < lay.slabs; ++sl) {
            i32x4 av[2][PL], bv[2][PL];
#pragma unroll
            for (int p = 0; p < PL; ++p)
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    if (i == 1 && !ox2) break;
                    const uint32_t* w = reinterpret_cast<const uint32_t*>(wr + (uint32_t)p * (uint32_t)crows * lay.wpitch +
                                                                          wal[i] + sl * 64u);
                    uint32_t d[5];
#pragma unroll
                    for (int h = 0; h < 5; ++h) d[h] = w[h];
#pragma unroll
                    for (int h = 0; h < 4; ++h) av[i][p][h] = (int)__builtin_amdgcn_alignbyte(d[h + 1], d[h], wsh[i]);
                }
#pragma unroll
            for (int p = 0; p < PL; ++p)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    if (j == 1 && !oy2) break;
                    bv[j][p] = *reinterpret_cast<const i32x4*>(rr + (uint32_t)p * srows * lay.rpitch + brow[j] + sl * 64u);
                }
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                if (i == 1 && !ox2) break;
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    if (j == 1 && !oy2) break;
                    acc[i][j][0] = __builtin_amdgcn_mfma_i32_16x16x64_i8(av[i][0], bv[j][0], acc[i][j][0], 0, 0, 0);
                    if constexpr (B == 2) {
                        acc[i][j][1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(av[i][0], bv[j][1], acc[i][j][1], 0, 0, 0);
                        acc[i][j][2] = __builtin_amdgcn_mfma_i32_16x16x64_i8(av[i][1], bv[j][1], acc[i][j][2], 0, 0, 0);
                        acc[i][j][1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(av[i][1], bv[j][0], acc[i][j][1], 0, 0, 0);
                    }
                }
            }
        }
    }
    __syncthreads();  // the box sums are there

    // ---- sum v^2 of every candidate, then each wave takes off twice its sum w * v
    for (uint32_t i = tid; i < (uint32_t)(orows * ocols); i += 256u) {
        long long v = 0;
#pragma unroll 4
        for (uint32_t dy = 0; dy < (uint32_t)crows; ++dy) v += rq[i + dy * (uint32_t)ocols];
        tot[i] = (unsigned long long)v;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const uint32_t oy = m16 + 16u * j;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t ox = 16u * i + 4u * kq + e;
                if (oy >= (uint32_t)orows || ox >= (uint32_t)ocols) continue;
                long long wv = acc[i][j][0][e];
                if constexpr (B == 2)
                    wv += ((long long)acc[i][j][B == 2 ? 2 : 0][e] << 16) + ((long long)acc[i][j][B == 2 ? 1 : 0][e] << 8);
                atomicAdd(tot + oy * (uint32_t)ocols + ox, (unsigned long long)(-2 * wv));
            }
        }
    __syncthreads();
    for (uint32_t i = tid; i < (uint32_t)(orows * ocols); i += 256u) {
        const uint32_t oy = i / (uint32_t)ocols, ox = i - oy * (uint32_t)ocols;
        atomicAdd(k.sums + (uint64_t)f * ssize * ssize + (uint64_t)(oy0 + oy) * ssize + ox0 + ox, tot[i]);
    }
}

template <int B>
__global__ void __launch_bounds__(256) shake_argmin_kernel(ShakeK k) {
    const uint32_t f = blockIdx.x;
    const int32_t ssize = 2 * k.s + 1, noff = ssize * ssize;
    __shared__ long long best_v[256];
    __shared__ int32_t best_i[256];
    long long bv = 0;
    int32_t bi = -1;
    for (int32_t o = threadIdx.x; o < noff; o += blockDim.x) {
        unsigned long long raw = k.sums[(uint64_t)f * noff + o] + k.sums[(uint64_t)k.n * noff];
        long long v = B == 1 ? (long long)(int32_t)(uint32_t)raw : (long long)raw;
        if (bi < 0 || v < bv) { bv = v; bi = o; }
    }
    best_v[threadIdx.x] = bv;
    best_i[threadIdx.x] = bi;
    __syncthreads();
    for (int32_t w = blockDim.x / 2; w > 0; w >>= 1) {
        if ((int32_t)threadIdx.x < w) {
            int32_t oi = best_i[threadIdx.x + w];
            long long ov = best_v[threadIdx.x + w];
            int32_t mi = best_i[threadIdx.x];
            long long mv = best_v[threadIdx.x];
            if (oi >= 0 && (mi < 0 || ov < mv || (ov == mv && oi < mi))) {
                best_i[threadIdx.x] = oi;
                best_v[threadIdx.x] = ov;
            }
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        int32_t b = f == 0 ? -1 : best_i[0];
        if (f == 0 || b < 0) {
            k.offsets[2 * f] = 0;
            k.offsets[2 * f + 1] = 0;
        } else {
            k.offsets[2 * f] = b % ssize - k.s;
            k.offsets[2 * f + 1] = b / ssize - k.s;
        }
    }
}

}  // namespace cp
