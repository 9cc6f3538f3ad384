// The tail of a bottleneck block of 8-bit convolutions, and the head of the next, as one launch: 3x3 convolution, 1x1 expansion,
// residual sum and, for the block behind it, the 1x1 reduction of the sum.
//
// As three launches the sum, four times as wide as what lies between, is written, read again by the reduction and a second time
// by the next sum, the 3x3 convolution's result is written and read, and on few images each launch is 4 to 5 us of start and
// end.  From the 3x3 convolution on nothing but a pixel's own values is needed, so a work-group takes 32 or 64 pixels in a row
// through all of it, and no pixel is computed twice.  us inside a recording, three launches and one, over 1, 8 and 64 images:
// 64 -> 256 -> 64 channels at 56x56 12.6 and 6.5, 17.7 and 10.2, 62.5 and 55.3; 128 -> 512 -> 128 at 28x28 12.1 and 7.5, 16.1
// and 8.6, 41.8 and 37.1; 256 -> 1024 -> 256 at 14x14 11.1 and 17.7 (not taken), 17.1 and 17.1, 35.6 and 25.3.
//
// The pixels that the taps fall on are one run of the dense image, which goes into LDS once (pixels an odd number of 16 bytes apart;
// taps outside the image read a pixel of zero points).  Weights are not shared between wavefronts: each has 32 channels of its own, for all of
// the tile's pixels or half of them, and reads their fragments from memory in the order that it uses them in (1 KB in a row), several
// steps ahead.  Rows of weights are permuted so that a lane ends with sixteen neighbouring channels of a pixel: a 16-byte
// store into the next convolution's operand, or into the result.  The residual is copied into LDS, where the sum replaces it in
// place and is the reduction's operand.  What bounds it: with 64 channels in between the vector instructions (11 per value of the sum, 5 per other value, and
// half as many again around them: 16 million in 46 us over 64 images of 56x56, with HBM's 128 MB a floor of 27 us beside them); with 256, one tile to a compute unit, the weights' way from L2 (1.1 MB to every
// compute unit, 41 bytes a cycle measured) and the phases that follow each other.  All results are those of the single calls, bit for bit: exact int32 sums, the same
// requantization (quant_math.h) and the same sum of codes (conv_device.h).
#include <algorithm>
#include <type_traits>

#include "contract.h"
#include "conv_device.h"
#include "bottleneck.h"

namespace chx {
namespace {

// async_copy16 from 32-bit offsets
__device__ __forceinline__ void async_copy16_at(const char* base, uint32_t offset, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(offset), "s"(base), "s"(lds_addr) : "memory", "m0");
}

// Sixteen sums of a pixel -> sixteen uint8 codes.
__device__ __forceinline__ v4i codes16(const v16i& sum, const float* scale, const QuantProduct& q) {
    float pre[16];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const v4f s = *reinterpret_cast<const v4f*>(scale + 4 * i);
#pragma unroll
        for (int e = 0; e < 4; ++e) pre[4 * i + e] = (float)sum[4 * i + e] * s[e];
    }
    if (q.path == 3) {  // (the path is the same in every lane)
#pragma unroll
        for (int e = 0; e < 16; ++e) pre[e] = quantize_prefloor_u8<3>(pre[e], q);
    } else {
#pragma unroll
        for (int e = 0; e < 16; ++e) pre[e] = quantize_prefloor_u8<1>(pre[e], q);
    }
    uint32_t word[4];
    floor_sat_u8x16(pre, word);
    return v4i{(int)word[0], (int)word[1], (int)word[2], (int)word[3]};
}

__device__ __forceinline__ v16i seeds16(const int32_t* add) {
    v16i acc;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const v4i v = *reinterpret_cast<const v4i*>(add + 4 * i);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[4 * i + e] = v[e];
    }
    return acc;
}

constexpr int kSigned = (int)0x80808080u;

// kMid: channels of the 3x3 convolution; kPT: tiles of 32 pixels; kWP: wavefronts that share them (kMid / 32 share the channels);
// kGroups: groups of kMid / 32 * kWP wavefronts, of which the first has the 3x3 convolution and each a share of the channels of the 1x1;
// kAffine: the sum has its short form, without a lower bound (ResidualAdd::affine is 1).
template <int kMid, int kPT, int kWP, int kGroups, bool kAffine>
__global__ __launch_bounds__(kMid * 2 * kWP * kGroups, 2) void bottleneck_kernel(BottleneckArgs) {
    constexpr int kWO = kMid / 32, kFirst = kWO * kWP, kWaves = kFirst * kGroups, kThreads = 64 * kWaves, kXT = kPT / kWP, kPx = 32 * kPT;
    constexpr int kSteps = kMid / 32, kTaps = kMid == 256 ? 1 : 3, kRing = kSteps * kTaps, kPitch = kMid + 16;
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const BottleneckArgs& a = kernel_arguments<BottleneckArgs>();
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, half = lane >> 5, wo = wave % kWO, wp = wave / kWO % kWP, group = wave / kFirst;
    const int tile = (int)(blockIdx.x & 7) * a.xcd_chunk + (int)(blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= a.xcd_chunk || tile >= a.tiles) return;
    const int m0 = tile * kPx, wide = a.wide, last_px = a.pixels - 1;
    const bool whole = m0 + kPx <= a.pixels;
    char* const patch = lds + kMid;  // behind a pixel of zero points
    char* const mids = lds + a.at_mid;
    char* const wides = lds + a.at_wide;
    float* const s_scale = reinterpret_cast<float*>(lds + a.at_table);
    const int rows = (kMid + wide + a.next + 63) & ~63;
    int32_t* const s_add = reinterpret_cast<int32_t*>(s_scale + rows);
    const uint32_t lane16 = (uint32_t)lane * 16u;
    auto fragment = [&](const char* base, int index) { return *reinterpret_cast<const v4i*>(base + (uint32_t)index * 1024u + lane16); };

    // ---- what is needed first: the pixels that the taps of the tile's pixels fall on, and the first weights ----
    const char* const w1 = a.w1 + (uint32_t)(wo * 9 * kSteps) * 1024u;
    v4i ring[kRing];
    {
        // a thread has one 16-byte chunk of every kRows-th pixel
        constexpr int kChunks = kMid / 16, kRows = kThreads / kChunks, kBatch = 3;
        const int first = m0 - a.W - 1, px0 = tid / kChunks, batches = a.patch_rows / kRows;
        const uint32_t from = __umul24((uint32_t)px0, (uint32_t)a.x_px) + (uint32_t)(tid % kChunks) * 16u;
        const bool inside = first >= 0 && first + a.patch_rows <= a.pixels;
        char* const to = patch + px0 * kPitch + (tid % kChunks) * 16;
        v4i v[kBatch];
        auto load = [&](int b0) {
            const char* row = a.x + (int64_t)(first + b0 * kRows) * a.x_px;
            if (inside) {
#pragma unroll
                for (int b = 0; b < kBatch; ++b) {
                    if (b0 + b < batches) v[b] = *reinterpret_cast<const v4i*>(row + from);
                    row += kRows * a.x_px;
                }
            } else {  // (pixels outside x are replaced: only taps outside the image look at them)
#pragma unroll
                for (int b = 0; b < kBatch; ++b) {
                    const int m = min(max(first + px0 + (b0 + b) * kRows, 0), last_px);
                    v[b] = *reinterpret_cast<const v4i*>(a.x + (int64_t)m * a.x_px + (tid % kChunks) * 16);
                }
            }
        };
        auto store = [&](int b0) {
#pragma unroll
            for (int b = 0; b < kBatch; ++b)
                if (b0 + b < batches) *reinterpret_cast<v4i*>(to + (b0 + b) * kRows * kPitch) = v[b] ^ (int)a.x_flip;
        };
        load(0);
        if (kGroups == 1 || group == 0) {
#pragma unroll
            for (int i = 0; i < kRing; ++i) ring[i] = fragment(w1, i);
        }
        // (64 rows of the tables are one convolution's)
        for (int i0 = wave * 64; i0 < rows; i0 += kThreads) {
            const bool one = i0 < kMid, two = i0 < kMid + wide;
            const float s = one ? a.s1 : two ? a.s2 : a.s3;
            const int corr = one ? a.corr1 : two ? a.corr2 : a.corr3;
            const v4i t = *reinterpret_cast<const v4i*>(reinterpret_cast<const char*>(a.table) + (uint32_t)i0 * 16u + lane16);
            s_scale[i0 + lane] = s * __int_as_float(t[0]);
            s_add[i0 + lane] = t[1] + __mul24(corr, t[2]);
        }
        if (tid < kChunks) *reinterpret_cast<v4i*>(lds + tid * 16) = v4i{a.fill, a.fill, a.fill, a.fill};
        store(0);
        for (int b0 = kBatch; b0 < batches; b0 += kBatch) {
            load(b0);
            store(b0);
        }
    }
    // the residual's pixels go where the sum's will be: chunk c of pixel p in place c ^ (p % 16) of its row
    {
        const int quads = a.quads_log2, copies = kPx / 4 << quads, most = last_px - m0;  // 256 bytes of a row for 16 lanes
        const char* const from = a.res.r + (int64_t)m0 * a.res.r_px_stride;
        for (int q = wave; q < copies; q += kWaves) {
            const int g = 4 * q + (lane >> 4), p = g >> quads, place = (g & ((1 << quads) - 1)) * 16 + ((lane & 15) ^ (p & 15));
            async_copy16_at(from, __umul24((uint32_t)min(p, most), (uint32_t)a.res.r_px_stride) + (uint32_t)place * 16u, (uint32_t)(uintptr_t)wides + (uint32_t)q * 1024u);
        }
    }
    int x_off[kXT];
    uint32_t taps[kXT];
#pragma unroll
    for (int j = 0; j < kXT; ++j) {
        const int p = (wp * kXT + j) * 32 + col;
        const uint32_t m = (uint32_t)min(m0 + p, last_px), row = fast_div(m, a.w_mul, a.w_shift), ow = m - row * (uint32_t)a.W;
        const uint32_t n = fast_div(row, a.h_mul, a.h_shift), oh = row - n * (uint32_t)a.H;
        const uint32_t cols = (ow > 0 ? 1u : 0u) | 2u | ((int)ow < a.W - 1 ? 4u : 0u);
        taps[j] = (oh > 0 ? cols : 0u) | cols << 3 | ((int)oh < a.H - 1 ? cols << 6 : 0u);
        x_off[j] = kMid + p * kPitch + 16 * half;
    }
    lds_barrier();

    // ---- 3x3 ----
    // The loops are in the order that they are written in (sched_barrier): left alone, the compiler moves a fragment's load in front of
    // its use.
    v16i acc[kPT];
    v4i expand[kSteps];
    const int first_wide = min(wave, (wide >> 5) - 1) * kSteps;
    if (kGroups == 1 || group == 0) {
        const v16i seed = seeds16(s_add + wo * 32 + 16 * half);
#pragma unroll
        for (int j = 0; j < kXT; ++j) acc[j] = seed;
        constexpr int kAhead = kMid == 256 ? 3 : 2, kRows = kAhead + 1;  // steps that the pixels are read ahead
        static_assert(kRing % kRows == 0 && kAhead <= kSteps, "");
        int tap = 0, tap_off = 0, kw = 0, off[kXT], off_next[kXT];
        int row_step = (a.W - 2) * kPitch;
        keep_scalar(row_step);
        auto offsets = [&](int (&to)[kXT]) {  // of tap `tap`, and on to the next (behind the last: the zero points)
#pragma unroll
            for (int j = 0; j < kXT; ++j) to[j] = (taps[j] >> tap) & 1 ? x_off[j] + tap_off : 16 * half;
            ++tap;
            kw = kw == 2 ? 0 : kw + 1;
            tap_off += kw == 0 ? row_step : kPitch;
        };
        v4i px[kRows][kXT];
        auto read = [&](v4i (&to)[kXT], const int (&from)[kXT], int k) {
#pragma unroll
            for (int j = 0; j < kXT; ++j) to[j] = *reinterpret_cast<const v4i*>(lds + from[j] + k * 32);
        };
        offsets(off);
#pragma unroll
        for (int k = 0; k < kAhead; ++k) read(px[k], off, k);  // (kAhead <= kSteps)
        auto taps_of = [&](auto last, int done) {
            const char* next = w1 + (uint32_t)(done * kSteps + kRing) * 1024u;
#pragma unroll
            for (int t = 0; t < kTaps; ++t) {
                offsets(off_next);
#pragma unroll
                for (int k = 0; k < kSteps; ++k) {
                    const int i = t * kSteps + k;
                    if (k + kAhead < kSteps) read(px[(i + kAhead) % kRows], off, k + kAhead);
                    else read(px[(i + kAhead) % kRows], off_next, k + kAhead - kSteps);
#pragma unroll
                    for (int j = 0; j < kXT; ++j) acc[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(ring[i], px[i % kRows][j], acc[j], 0, 0, 0);
                    if constexpr (decltype(last)::value) {
                        if (t == 0) expand[k] = fragment(a.w2, first_wide + k);
                    } else {
                        ring[i] = fragment(next, i);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int j = 0; j < kXT; ++j) off[j] = off_next[j];
            }
        };
#pragma unroll 1
        for (int done = 0; done < 9 - kTaps; done += kTaps) taps_of(std::false_type(), done);
        taps_of(std::true_type(), 9 - kTaps);
        const QuantProduct q1 = in_vector_registers(a.q1);
#pragma unroll
        for (int j = 0; j < kXT; ++j) {
            const v4i codes = codes16(acc[j], s_scale + wo * 32 + 16 * half, q1);
            *reinterpret_cast<v4i*>(mids + ((wp * kXT + j) * 32 + col) * kPitch + wo * 32 + 16 * half) = codes ^ kSigned;
        }
    } else {  // (the second group only brings what the first needs, until the expansion)
#pragma unroll
        for (int k = 0; k < kSteps; ++k) expand[k] = fragment(a.w2, first_wide + k);
    }
    wait_vmcnt<0>();  // (the residual is there, too)
    lds_barrier();

    // ---- 1x1 expansion and the sum: every wavefront has all pixels, and channels of its own ----
    const int wide_tiles = wide >> 5, reduce_steps = wide >> 5;
    const char* const w3 = a.w3 + (uint32_t)(min(wo + kWO * group, max((a.next >> 5) - 1, 0)) * reduce_steps) * 1024u;
    v4i reduce[8];
    {
        const QuantProduct q2 = in_vector_registers(a.q2);
        ResidualAdd res = a.res;
        if constexpr (kAffine) res = in_vector_registers(a.res);
        const int flip = kSigned ^ (int)a.y_flip;
        const int64_t y_px = a.y_px;
        char* const y = a.y + (int64_t)m0 * y_px;
        const uint32_t y_lane = __umul24((uint32_t)col, (uint32_t)y_px) + 16u * (uint32_t)half;
        v4i px[kSteps][kPT];
#pragma unroll
        for (int k = 0; k < kSteps; ++k)
#pragma unroll
            for (int j = 0; j < kPT; ++j) px[k][j] = *reinterpret_cast<const v4i*>(mids + (j * 32 + col) * kPitch + 16 * half + k * 32);
#pragma unroll 1
        for (int t = wave; t < wide_tiles; t += kWaves) {
            const float* const scale = s_scale + kMid + t * 32 + 16 * half;
            {
                const v16i seed = seeds16(s_add + kMid + t * 32 + 16 * half);
#pragma unroll
                for (int j = 0; j < kPT; ++j) acc[j] = seed;
            }
            const int next = min(t + kWaves, wide_tiles - 1) * kSteps;
#pragma unroll
            for (int k = 0; k < kSteps; ++k) {
#pragma unroll
                for (int j = 0; j < kPT; ++j) acc[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(expand[k], px[k][j], acc[j], 0, 0, 0);
                expand[k] = fragment(a.w2, next + k);
                __builtin_amdgcn_sched_barrier(0);
            }
            char* const at = wides + col * wide + ((((2 * t + half) & ~15) | (((2 * t + half) & 15) ^ (col & 15))) << 4);
#pragma unroll
            for (int j = 0; j < kPT; ++j) {
                v4i* const place = reinterpret_cast<v4i*>(at + j * 32 * wide);
                const v4i r = *place;
                v4i codes = codes16(acc[j], scale, q2);
                if constexpr (kAffine) codes = affine_residual16<false>(codes, r, res);
                else if (res.affine == 2) codes = affine_residual16<true>(codes, r, res);
                else codes = add_residual16_any(codes, r, res);
                codes ^= kSigned;
                *place = codes;
                char* const row = y + j * 32 * y_px + t * 32;
                codes ^= flip;
                if (whole) *reinterpret_cast<v4i*>(row + y_lane) = codes;
                else if (m0 + j * 32 + col <= last_px) *reinterpret_cast<v4i*>(row + y_lane) = codes;
            }
        }
    }
    if (a.z) {
#pragma unroll
        for (int k = 0; k < 8; ++k) reduce[k] = fragment(w3, k);
    }
    lds_barrier();

    // ---- 1x1 reduction for the next block ----
    if (a.z) {
        constexpr int kAhead = 3, kRows = 4;
        const QuantProduct q3 = in_vector_registers(a.q3);
        const int swizzle = (half ^ (col & 15)) << 4, z_flip = (int)a.z_flip;
        const int64_t z_px = a.z_px;
        char* const z = a.z + (int64_t)(m0 + wp * kXT * 32) * z_px;
        const uint32_t z_lane = __umul24((uint32_t)col, (uint32_t)z_px) + 16u * (uint32_t)half;
        const char* const from = wides + (wp * kXT * 32 + col) * wide;
#pragma unroll 1
        for (int t = wo + kWO * group; t < a.next >> 5; t += kWO * kGroups) {
            {
                const v16i seed = seeds16(s_add + kMid + wide + t * 32 + 16 * half);
#pragma unroll
                for (int j = 0; j < kXT; ++j) acc[j] = seed;
            }
            const char* w = a.w3 + (uint32_t)(t * reduce_steps) * 1024u;
            v4i px[kRows][kXT];
            auto read = [&](v4i (&to)[kXT], const char* row, int k) {
#pragma unroll
                for (int j = 0; j < kXT; ++j) to[j] = *reinterpret_cast<const v4i*>(row + j * 32 * wide + (swizzle ^ (k * 32)));
            };
#pragma unroll
            for (int k = 0; k < kAhead; ++k) read(px[k], from, k);
#pragma unroll 1
            for (int s = 0; s < reduce_steps; s += 8) {
                // (behind the tile's last steps: the next tile's first, or some again)
                const int ahead = s + 8 < reduce_steps ? s + 8 : t + kWO * kGroups < a.next >> 5 ? kWO * kGroups * reduce_steps : 0;
                const char *const row = from + s * 32, *const row_next = from + (s + 8 < reduce_steps ? s + 8 : 0) * 32;
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    read(px[(k + kAhead) % kRows], k + kAhead < 8 ? row : row_next, (k + kAhead) % 8);
#pragma unroll
                    for (int j = 0; j < kXT; ++j) acc[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(reduce[k], px[k % kRows][j], acc[j], 0, 0, 0);
                    reduce[k] = fragment(w, ahead + k);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
#pragma unroll
            for (int j = 0; j < kXT; ++j) {
                const v4i codes = codes16(acc[j], s_scale + kMid + wide + t * 32 + 16 * half, q3) ^ z_flip;
                char* const row = z + j * 32 * z_px + t * 32;
                if (whole) *reinterpret_cast<v4i*>(row + z_lane) = codes;
                else if (m0 + (wp * kXT + j) * 32 + col <= last_px) *reinterpret_cast<v4i*>(row + z_lane) = codes;
            }
        }
    }
}

// A wavefront per (K step, 32 rows); K in the order (kh, kw, c).
__global__ __launch_bounds__(64) void pack_bottleneck_kernel(const int8_t* w, int64_t s_row, int64_t s_c, int64_t s_h, int64_t s_w, int C, int KW, char* fragments) {
    const int lane = threadIdx.x, step = (int)blockIdx.x, steps = (int)gridDim.x, tile = (int)blockIdx.y;
    const int k0 = step * 32 + (lane >> 5) * 16, tap = k0 / C, c0 = k0 - tap * C, kh = tap / KW, kw = tap - kh * KW;  // (C is a multiple of 32)
    const int8_t* from = w + (tile * 32 + channel_of(lane & 31)) * s_row + c0 * s_c + kh * s_h + kw * s_w;
    v4i v = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i / 4] |= (int)((uint32_t)(uint8_t)from[i * s_c] << (8 * (i % 4)));
    *reinterpret_cast<v4i*>(fragments + ((int64_t)tile * steps + step) * 1024 + lane * 16) = v;
}

// A wavefront per row.
__global__ __launch_bounds__(64) void pack_bottleneck_table_kernel(const int8_t* w, int64_t s_row, int64_t s_c, int64_t s_h, int64_t s_w, int C, int KH, int KW, const char* scale, int64_t s_scale,
                                                                   const char* bias, int64_t s_bias, int32_t* table) {
    const int row = (int)blockIdx.x;
    int32_t sum = 0;
    for (int kh = 0; kh < KH; ++kh)
        for (int kw = 0; kw < KW; ++kw)
            for (int c = threadIdx.x; c < C; c += 64) sum += w[row * s_row + c * s_c + kh * s_h + kw * s_w];
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) sum += __shfl_xor(sum, d);
    if (threadIdx.x == 0) {
        const int32_t s = *reinterpret_cast<const int32_t*>(scale + row * s_scale), b = bias ? *reinterpret_cast<const int32_t*>(bias + row * s_bias) : 0;
        *reinterpret_cast<v4i*>(table + row * 4) = v4i{s, b, sum, 0};
    }
}

constexpr int kLdsOfUnit = 160 * 1024;

int lay_out(BottleneckArgs& a, int px_tiles, int px_waves, int groups) {
    const int px = 32 * px_tiles;
    a.px_tiles = px_tiles;
    a.px_waves = px_waves;
    a.groups = groups;
    const int rows = 64 * (a.mid / 32 * px_waves * groups) / (a.mid / 16);  // that a work-group brings at a time
    a.patch_rows = (px + 2 * a.W + 2 + rows - 1) / rows * rows;
    a.at_mid = a.mid + a.patch_rows * (a.mid + 16);
    a.at_wide = a.at_mid + px * (a.mid + 16);
    a.at_table = a.at_wide + px * a.wide;
    return a.at_table + (a.mid + a.wide + a.next + 63) / 64 * 64 * 8;
}

template <int kMid, int kPT, int kWP, int kGroups, bool kAffine>
int launch(const BottleneckArgs& a, hipStream_t s) {
    if (a.lds > 64 * 1024)  // (has to be asked for, on every device)
        CHX_HIP_CALL(hipFuncSetAttribute(reinterpret_cast<const void*>(&bottleneck_kernel<kMid, kPT, kWP, kGroups, kAffine>), hipFuncAttributeMaxDynamicSharedMemorySize, kLdsOfUnit));
    bottleneck_kernel<kMid, kPT, kWP, kGroups, kAffine><<<8 * a.xcd_chunk, kMid * 2 * kWP * kGroups, a.lds, s>>>(a);
    return launch_check("bottleneck_kernel");
}

}  // namespace

int plan_bottleneck(BottleneckArgs* launch) {
    BottleneckArgs& a = *launch;
    // Pixels of a work-group, and whether the block is one launch: by 400 drawn blocks measured both ways inside a recording, three
    // with weights of their own in turn.  Few pixels leave compute units idle when they are shared out in tiles of 64, and each
    // work-group reads all weights for its tile.  256 channels on few pixels are faster as single launches (up to 1.4 times).  With 256 a tile takes 16 to 18 us however few
    // there are.  256 -> 1024 -> 256, six in a row, one launch and three: inside a recording 18.3 and 16.7 us at 980 pixels, 18.3 and 17.9 at 1,176 and
    // 1,372, 18.2 and 18.2 at 1,568, 18.2 and 18.8 at 1,960, 18.3 and 20.3 at 2,352; run by run, where a launch costs more, 24.5 and 22.8 at 588, 24.5 and
    // 26.3 at 784, 25.5 and 29.4 at 1,372.  The line is that of recordings, which are what is run again and again; run by run
    // 2 to 4 us a block are left between 700 pixels and it.  Two launches without a reduction, and three with one to more than 256
    // channels, meet the one at 2,500.
    const int fewest = a.next == 0 || a.next > 256 ? 2500 : 1500;
    if (a.W >= 8192) CHX_FAIL(CHX_HIP_EUNSUPPORTED, "bottleneck: the rows do not fit");  // (some 950 pixels of 64 channels do; what follows counts bytes in 32 bits)
    if (a.mid == 256 && (a.pixels < fewest || a.pixels > 60000)) CHX_FAIL(CHX_HIP_EUNSUPPORTED, "bottleneck: slower than its convolutions");
    const int pt = a.mid == 64 ? 2 : a.mid == 128 ? (a.pixels < 24000 ? 1 : 2) : a.pixels < 9000 ? 1 : 2, wp = a.mid == 64 ? 2 : 1;
    // A second group of wavefronts: where a compute unit has at most two tiles, one group leaves its four SIMDs waiting for weights in
    // the 1x1 convolutions.  Inside a recording, with one group and with two: 64 channels 8.2 and 7.5 us at 245 tiles, 10.8 and 10.5
    // at 490, 13.3 and 15.3 at 588; 128 channels 9.5 and 8.5 at 245, 13.7 and 13.6 at 490 (without a reduction 11.9 and 11.3), 17.7
    // and 19.1 at 588.  Four groups of 128 channels are no faster than two (8.8 and 8.6 at 196 tiles), and with 256 channels, where
    // a group has eight wavefronts, two are slower at every size (17.7 and 16.7 at 49 tiles, 34.5 and 31.7 at 392).
    a.tiles = (a.pixels + 32 * pt - 1) / (32 * pt);
    a.lds = lay_out(a, pt, wp, a.mid < 256 && pt == wp && a.tiles <= 512 ? 2 : 1);
    if (a.groups == 2 && a.lds * (a.tiles > 256 ? 2 : 1) > kLdsOfUnit) a.lds = lay_out(a, pt, wp, 1);  // (its patch may be larger)
    if (a.lds > kLdsOfUnit) CHX_FAIL(CHX_HIP_EUNSUPPORTED, "bottleneck: the rows do not fit");
    a.xcd_chunk = (a.tiles + 7) / 8;
    magic_divisor((uint32_t)a.W, &a.w_mul, &a.w_shift);
    magic_divisor((uint32_t)a.H, &a.h_mul, &a.h_shift);
    a.quads_log2 = 0;
    while (256 << a.quads_log2 < a.wide) ++a.quads_log2;
    return CHX_HIP_OK;
}

int launch_bottleneck(const BottleneckArgs& a, hipStream_t s) {
#define CHX_SPLIT(MID, PT, WP, GROUPS)                                                                                   \
    if (a.mid == MID && a.px_tiles == PT && a.px_waves == WP && a.groups == GROUPS)                                         \
        return a.res.affine == 1 ? launch<MID, PT, WP, GROUPS, true>(a, s) : launch<MID, PT, WP, GROUPS, false>(a, s);
    CHX_SPLIT(64, 2, 2, 1)
    CHX_SPLIT(64, 2, 2, 2)
    CHX_SPLIT(128, 1, 1, 1)
    CHX_SPLIT(128, 1, 1, 2)
    CHX_SPLIT(128, 2, 1, 1)
    CHX_SPLIT(256, 1, 1, 1)
    CHX_SPLIT(256, 2, 1, 1)
#undef CHX_SPLIT
    CHX_FAIL(CHX_HIP_EINVAL, "bottleneck: no kernel for %d channels and %d tiles of pixels", a.mid, a.px_tiles);
}

int pack_bottleneck(const chx_hip_tensor& w, const chx_hip_tensor& scale, const chx_hip_tensor* bias, char* fragments, int32_t* table, hipStream_t s) {
    const int rows = (int)w.shape[0], C = (int)w.shape[1], KH = (int)w.shape[2], KW = (int)w.shape[3];
    const int8_t* data = static_cast<const int8_t*>(w.data);
    pack_bottleneck_kernel<<<dim3((unsigned)(KH * KW * C / 32), (unsigned)(rows / 32)), 64, 0, s>>>(data, w.strides[0], w.strides[1], w.strides[2], w.strides[3], C, KW, fragments);
    CHX_PROPAGATE(launch_check("pack_bottleneck_kernel"));
    pack_bottleneck_table_kernel<<<(unsigned)rows, 64, 0, s>>>(data, w.strides[0], w.strides[1], w.strides[2], w.strides[3], C, KH, KW, static_cast<const char*>(scale.data),
                                                             numel(scale) > 1 ? scale.strides[0] : 0, bias ? static_cast<const char*>(bias->data) : nullptr, bias ? bias->strides[0] : 0, table);
    return launch_check("pack_bottleneck_table_kernel");
}

}  // namespace chx
