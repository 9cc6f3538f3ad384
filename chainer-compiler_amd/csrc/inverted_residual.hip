// An inverted residual block of 8-bit convolutions as one launch: 1x1 expansion, depthwise 3x3, 1x1 projection, residual sum.
//
// As three launches the expanded activations, six times the block's input, are written and read twice: 420 of 460 MB
// for 16 -> 96 -> 24 channels over 128 images of 112x112, and on one image the block is three launches of 3.5 us with a
// boundary each.  Here a work-group takes a strip of R output rows of an image, whole width, and walks through the expanded
// channels in chunks of 32 or 64.  In one interval its eight wavefronts do three things, each for another chunk, with one
// barrier at the end: expand chunk i into LDS, convolve chunk i - 1 depthwise from LDS into LDS, and multiply chunk i - 2
// into the projection's sums, which stay in registers.  Wide images take one buffer each for the expanded and the convolved chunk
// instead of two, which leaves room for more rows: then an interval is the expansion of chunk i and the projection of chunk i - 1,
// a barrier, the depthwise part of chunk i, a barrier.  In us, as three launches inside a graph and as one, over 1, 32 and
// 128 images: 16 -> 96 -> 24 channels, 112x112 to 56x56, 14.1 and 8.1, 34.8 and 20.0, 97.1 and 66.8; 32 -> 192 -> 32 at
// 28x28 14.2 and 7.2, 18.0 and 10.8, 37.4 and 20.2; 64 -> 384 -> 64 at 14x14 14.0 and 7.8, 17.0 and 9.1, 24.5 and 16.9;
// 160 -> 960 -> 160 at 7x7 13.9 and 12.7, 15.7 and 13.7, 30.3 and 17.1.
//
// What bounds it is vector instructions (their pipeline is 0.8 full on 128 images of 112x112 and 56x56; 0.4 at 7x7, where a work-group has the compute unit
// alone and waits at its barriers): 5 per requantized value (conversion, scale, two multiply-adds, conversion), 4.5
// dot products and shifts per depthwise result, so the layouts are chosen to need none for moving data:
//  * Expansion: the pixels are the rows of the MFMA, so that a lane holds one channel, its scale and its zero point's
//    share for the whole interval, and, with the pixels in the order of pixel_of(), sixteen neighbouring pixels: one
//    16-byte store into LDS [channel][pixel].  Rows of pixels follow each other with at least one pixel between them
//    that is the padding on the right of one and on the left of the next; outside the image a mask puts the zero point.
//  * Depthwise: a lane has one channel; v_dot4 takes three neighbouring bytes of a row against a filter row.  Of four
//    results two read an aligned dword (against the filter row, or the filter row moved up by a byte), two a shifted one.
//  * Projection: its operand is wanted [pixel][channel]: ds_read_b64_tr_b8 transposes 8 x 16 bytes on the way from LDS.
//  * The projection's filters are permuted so that a lane ends with sixteen neighbouring channels of a pixel: one store.
// The input strip lies in LDS with pixels an odd number of 16 bytes apart, channels of the other buffers likewise, so that 16-byte accesses keep
// off each other's banks (the depthwise part's dwords share a fourth of them: 3.5 to 6.7 conflict cycles per LDS instruction in all).  All results are those of the three convolutions and the sum, bit for bit: exact int32 sums, the same
// requantization (quant_math.h) and the same sum of codes (conv_device.h).
#include <algorithm>
#include <cstring>

#include "contract.h"
#include "conv_device.h"
#include "inverted_residual.h"

namespace chx {
namespace {

constexpr int kWaves = 8, kMostTiles = 3;

typedef int v2i __attribute__((ext_vector_type(2)));
typedef int v16i __attribute__((ext_vector_type(16)));

// The pixel of a run of 32 that row m of the expansion's MFMA takes: register r of lane half h is row
// 8 (r / 4) + 4 h + r % 4, and should be pixel 16 h + r.  (The projection's channels likewise.)
__host__ __device__ __forceinline__ int pixel_of(int m) {
    return 16 * ((m >> 2) & 1) + 4 * (m >> 3) + (m & 3);
}

__device__ __forceinline__ v2i transposed8(uint32_t lds_address) {
    typedef __attribute__((address_space(3))) v2i* Lds;
    return __builtin_amdgcn_ds_read_tr8_b64_v2i32((Lds)lds_address);
}

// The codes' values in front of the conversion; the path is the same in every lane.
template <int kCount>
__device__ __forceinline__ void prefloor(float (&v)[kCount], const QuantProduct& q) {
    if (q.path == 3) {
#pragma unroll
        for (int e = 0; e < kCount; ++e) v[e] = quantize_prefloor_u8<3>(v[e], q);
    } else {
#pragma unroll
        for (int e = 0; e < kCount; ++e) v[e] = quantize_prefloor_u8<1>(v[e], q);
    }
}

// the first `n` of sixteen bytes
__device__ __forceinline__ void store_first(char* dst, v4i v, int n) {
    for (int e = 0; e < n; ++e) dst[e] = (char)((uint32_t)v[e / 4] >> (8 * (e % 4)));
}

// kTiles: 32 x 32 tiles of the projection per wavefront, at most; kG: tiles of 32 expanded channels per interval; kKS: K steps
// of the expansion; kBuffers: of the expanded and of the convolved channels.
template <int kStride, int kTiles, int kG, int kKS, int kBuffers>
__global__ __launch_bounds__(64 * kWaves, (kTiles == 1 || (kTiles == 2 && kBuffers == 1)) && kG <= 2 ? 4 : 2) void inverted_residual_kernel(InvertedResidualArgs) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const InvertedResidualArgs& a = kernel_arguments<InvertedResidualArgs>();
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, half = lane >> 5;
    // an XCD takes a contiguous run of strips: neighbours share input rows
    const int block = (int)(blockIdx.x & 7) * a.xcd_chunk + (int)(blockIdx.x >> 3);
    if (block >= a.blocks) return;
    const int n = (int)fast_div((uint32_t)block, a.strips_mul, a.strips_shift), oh0 = (block - n * a.strips) * a.R, ih0 = oh0 * kStride - 1;
    char* const xs = lds;
    char* const mask = lds + a.at_mask;
    char* const hid = lds + a.at_hid;  // [2][kG * 32][cs], a channel's pixels from byte 16 on
    char* const dw = lds + a.at_dw;    // [2][kG * 32][cs2]
    float* const s_scale = reinterpret_cast<float*>(lds + a.at_t3);
    int32_t* const s_add = reinterpret_cast<int32_t*>(s_scale + 32 * a.tiles_oc);

    // this wavefront's tile of 32 expanded channels in every interval, and its share of the runs and items
    constexpr int kShare = kWaves / kG;
    const int g = wave % kG, share = wave / kG;
    const int runs = a.pixels >> 5;

    // What the loop reads of the arguments, in registers: where a field is used behind a branch it would be fetched there.
    const int intervals = a.intervals, cs = a.cs, cs2 = a.cs2, pitch = a.pitch, pitch_o = a.pitch_o, blocks = pitch_o >> 3, items = a.items, px_bytes = a.px_bytes;
    const int corr1 = a.corr1, corr2 = a.corr2, fill = a.fill, last_chunk = (a.x_chunks - 1) * 16, tiles = a.tiles_px * a.tiles_oc;
    const uint32_t blk_mul = a.blk_mul, blk_shift = a.blk_shift;
    const float s1 = a.s1, s2 = a.s2;
    const QuantProduct q1 = in_vector_registers(a.q1), q2 = in_vector_registers(a.q2);
    const char* const w1_base = a.w1 + (int64_t)g * kKS * 1024 + lane * 16;
    const int32_t* const t1_base = a.t1 + (g * 32 + col) * 4;
    const int32_t* const t2_base = a.t2 + (g * 32 + col) * 8;

    v4i w1[kKS], c1;  // of the chunk to be expanded next, and its table
    auto fetch1 = [&](int chunk) __attribute__((always_inline)) {
        const char* w = w1_base + (int64_t)chunk * kG * kKS * 1024;
#pragma unroll
        for (int k = 0; k < kKS; ++k) w1[k] = *reinterpret_cast<const v4i*>(w + k * 1024);
        c1 = *reinterpret_cast<const v4i*>(t1_base + chunk * kG * 128);
    };
    fetch1(0);

    // ---- the input strip, and what the other buffers need once ----
    {
        // A strip's rows lie behind each other, so that a chunk's place in memory is its number but for what lies between two
        // pixels' chunks; in LDS there is room behind each pixel and each row.  Rows outside the image are masked later: what is read for them is
        // the nearest chunk inside.  (Divisions for each chunk's row and pixel, four chunks at a time, were 110 of a wavefront's 1,380 vector
        // instructions for 16 -> 96 -> 24 at 112x112: 77.8 us for 75.8.)
        constexpr int kBatch = 2;  // chunks requested before the first is stored
        const int per_row = a.W * a.x_chunks, total = a.rows * per_row, first = ih0 * per_row, most = a.H * per_row - 1;
        const int px_room = a.px_bytes - 16 * a.x_chunks, x_room = (int)a.x_px - 16 * a.x_chunks, row_room = (a.pitch - a.W) * a.px_bytes;
        const char* x = a.x + (int64_t)n * a.x_n;
        for (int i0 = tid; i0 < total; i0 += kBatch * 64 * kWaves) {
            v4i v[kBatch];
            int at[kBatch];
#pragma unroll
            for (int b = 0; b < kBatch; ++b) {
                const int i = min(i0 + b * 64 * kWaves, total - 1);
                const int chunk = min(max(first + i, 0), most);
                uint32_t from = (uint32_t)chunk * 16;
                if (x_room != 0) from += fast_div((uint32_t)chunk, a.chunks_mul, a.chunks_shift) * (uint32_t)x_room;
                v[b] = *reinterpret_cast<const v4i*>(x + from);
                at[b] = i * 16 + (int)fast_div((uint32_t)i, a.row_mul, a.row_shift) * row_room;
                if (px_room != 0) at[b] += (int)fast_div((uint32_t)i, a.chunks_mul, a.chunks_shift) * px_room;
            }
#pragma unroll
            for (int b = 0; b < kBatch; ++b) *reinterpret_cast<v4i*>(xs + at[b]) = v[b] ^ (int)a.x_flip;
        }
        for (int p = tid * 4; p < a.pixels; p += 4 * 64 * kWaves) {  // (a row's pitch is a multiple of 4)
            const int row = (int)fast_div((uint32_t)p, a.pitch_mul, a.pitch_shift), xx = p - row * a.pitch, ih = ih0 + row;
            const int left = ih >= 0 && ih < a.H ? min(max(a.W - xx, 0), 4) : 0;
            *reinterpret_cast<uint32_t*>(mask + p) = left == 0 ? 0u : 0xffffffffu >> (32 - 8 * left);
        }
        for (int i = tid; i < kBuffers * kG * 32; i += 64 * kWaves) *reinterpret_cast<v4i*>(hid + i * a.cs) = v4i{a.fill, a.fill, a.fill, a.fill};
        for (int i = tid; i < 32 * a.tiles_oc; i += 64 * kWaves) {
            const v4i t = *reinterpret_cast<const v4i*>(a.t3 + i * 4);
            s_scale[i] = a.s3 * __int_as_float(t[0]);
            s_add[i] = t[1] + a.corr3 * t[2];
        }
    }
    __syncthreads();

    v16i acc[kTiles];
    int tile_oc[kTiles], tile_px[kTiles];
    const char* w3_at[kTiles];
#pragma unroll
    for (int t = 0; t < kTiles; ++t) {
        const int i = min(wave + kWaves * t, tiles - 1);
        tile_px[t] = (int)fast_div((uint32_t)i, a.oct_mul, a.oct_shift);
        tile_oc[t] = i - tile_px[t] * a.tiles_oc;
        w3_at[t] = a.w3 + (int64_t)tile_oc[t] * a.hid_tiles_padded * 1024 + lane * 16;
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[t][r] = 0;
    }

    const int cs_chunk = kG * 32 * cs, cs2_chunk = kG * 32 * cs2;
    const char* const px0 = xs + pixel_of(col) * px_bytes;
    char* const hid_lane = hid + (g * 32 + col) * cs;
    char* const dw_lane = dw + (g * 32 + col) * cs2;
    // lanes of a group of 16 read 8 channels of 16 pixels, two to a channel, and hold 8 channels of a pixel
    const int in = lane & 15, quarter = lane >> 4;
    const uint32_t dw_from = (uint32_t)(uintptr_t)dw + (uint32_t)((16 * (quarter >> 1) + (in >> 1)) * cs2 + 16 * (quarter & 1) + 8 * (in & 1));
    auto expand = [&](char* to) __attribute__((always_inline)) {
        const float scale = s1 * __int_as_float(c1[0]);
        const int32_t add = c1[1] + corr1 * c1[2];
        to += 16 + 16 * half;
        for (int run = share; run < runs; run += kShare) {
            const char* px = px0 + run * 32 * px_bytes;
            v4i x[kKS];
#pragma unroll
            for (int k = 0; k < kKS; ++k) x[k] = *reinterpret_cast<const v4i*>(px + min(k * 32 + 16 * half, last_chunk));
            const v4i m = *reinterpret_cast<const v4i*>(mask + run * 32 + 16 * half);
            v16i sum;
#pragma unroll
            for (int r = 0; r < 16; ++r) sum[r] = add;
#pragma unroll
            for (int k = 0; k < kKS; ++k) sum = __builtin_amdgcn_mfma_i32_32x32x32_i8(x[k], w1[k], sum, 0, 0, 0);
            float pre[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) pre[r] = (float)sum[r] * scale;
            prefloor(pre, q1);
            uint32_t word[4];
            floor_sat_u8x16(pre, word);
            v4i out;
#pragma unroll
            for (int e = 0; e < 4; ++e) out[e] = ((int)(word[e] ^ 0x80808080u) & m[e]) | (fill & ~m[e]);
            *reinterpret_cast<v4i*>(to + run * 32) = out;
        }
    };
    auto depthwise = [&](v4i d0, v2i d1, const char* from, char* to) __attribute__((always_inline)) {
        const float scale = s2 * __int_as_float(d0[3]);
        const int32_t add = d1[0] + corr2 * d1[1];
        from += 12;  // the dword in front of the first pixel
        const int w[3] = {d0[0], d0[1], d0[2]}, wu[3] = {d0[0] << 8, d0[1] << 8, d0[2] << 8};
        for (int item0 = share * 2; item0 < items; item0 += kShare * 2) {
            const int item = min(item0 + half, items - 1);
            const int r = (int)fast_div((uint32_t)item, blk_mul, blk_shift), xb = item - r * blocks;
            const char* src = from + r * kStride * pitch + xb * 8 * kStride;
            int32_t sum[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) sum[e] = add;
#pragma unroll
            for (int f = 0; f < 3; ++f) {
                const uint32_t* row = reinterpret_cast<const uint32_t*>(src + f * pitch);
                auto dot = [&](int e, uint32_t v, int weights) __attribute__((always_inline)) { sum[e] = __builtin_amdgcn_sdot4((int)v, weights, sum[e], false); };
                if constexpr (kStride == 1) {
                    const uint32_t b = row[0], p = row[1], q1 = row[2], nx = row[3];
                    dot(0, __builtin_amdgcn_alignbyte(p, b, 3), w[f]);
                    dot(1, p, w[f]);
                    dot(2, p, wu[f]);
                    dot(3, __builtin_amdgcn_alignbyte(q1, p, 2), w[f]);
                    dot(4, __builtin_amdgcn_alignbyte(q1, p, 3), w[f]);
                    dot(5, q1, w[f]);
                    dot(6, q1, wu[f]);
                    dot(7, __builtin_amdgcn_alignbyte(nx, q1, 2), w[f]);
                } else {
                    uint32_t v[5];
#pragma unroll
                    for (int e = 0; e < 5; ++e) v[e] = row[e];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        dot(2 * e, __builtin_amdgcn_alignbyte(v[e + 1], v[e], 3), w[f]);
                        dot(2 * e + 1, v[e + 1], wu[f]);
                    }
                }
            }
            float pre[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) pre[e] = (float)sum[e] * scale;
            prefloor(pre, q2);
            uint32_t lo, hi;
            floor_sat_u8x8(pre, &lo, &hi);
            *reinterpret_cast<v2i*>(to + r * pitch_o + xb * 8) = v2i{(int)(lo ^ 0x80808080u), (int)(hi ^ 0x80808080u)};
        }
    };
    v4i w3[kTiles][kG];  // the projection's filters for a chunk
    auto fetch3 = [&](int chunk) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < kTiles; ++t)
#pragma unroll
            for (int k = 0; k < kG; ++k) w3[t][k] = *reinterpret_cast<const v4i*>(w3_at[t] + (chunk * kG + k) * 1024);
    };
    auto project = [&](uint32_t from) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < kTiles; ++t) {
            if (wave + kWaves * t >= tiles) break;
            v2i lo[kG], hi[kG];
#pragma unroll
            for (int k = 0; k < kG; ++k) {
                const uint32_t at = from + (uint32_t)(k * 32 * cs2 + tile_px[t] * 32);
                lo[k] = transposed8(at);
                hi[k] = transposed8(at + 8 * (uint32_t)cs2);
            }
#pragma unroll
            for (int k = 0; k < kG; ++k) acc[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(w3[t][k], v4i{lo[k][0], lo[k][1], hi[k][0], hi[k][1]}, acc[t], 0, 0, 0);
        }
    };
    auto fetch2 = [&](int chunk, v4i* d0, v2i* d1) __attribute__((always_inline)) {
        const int32_t* t2 = t2_base + chunk * kG * 256;
        *d0 = *reinterpret_cast<const v4i*>(t2);
        *d1 = *reinterpret_cast<const v2i*>(t2 + 4);
    };
    // Memory is read without a branch around it (at the ends: some chunk again), or the compiler waits for everything
    // where the branches meet.  The fragments of this interval's expansion are there first; the filters of its second and
    // third part are requested then, and the next expansion's behind this one.
    auto expansion_is_there = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < kKS; ++k) asm volatile("" : "+v"(w1[k]));
        asm volatile("" : "+v"(c1));
    };
    v4i d0;
    v2i d1;
    if constexpr (kBuffers == 2) {
        for (int i = 0; i < intervals + 2; ++i) {
            expansion_is_there();
            fetch2(min(max(i - 1, 0), intervals - 1), &d0, &d1);
            fetch3(min(max(i - 2, 0), intervals - 1));
            if (i < intervals) expand(hid_lane + (i & 1) * cs_chunk);
            fetch1(min(i + 1, intervals - 1));
            if (i >= 1 && i <= intervals) depthwise(d0, d1, hid_lane + ((i - 1) & 1) * cs_chunk, dw_lane + ((i - 1) & 1) * cs2_chunk);
            if (i >= 2) project(dw_from + (uint32_t)((i & 1) * cs2_chunk));
            __syncthreads();
        }
    } else {
        for (int i = 0;; ++i) {
            expansion_is_there();
            if (kTiles == 1) fetch3(max(i - 1, 0));
            if (i < intervals) expand(hid_lane);
            if (kTiles != 1) fetch3(max(i - 1, 0));  // (in front of the expansion they are registers too many)
            fetch2(min(i, intervals - 1), &d0, &d1);
            fetch1(min(i + 1, intervals - 1));
            if (i >= 1) project(dw_from);
            if (i == intervals) break;
            __syncthreads();
            depthwise(d0, d1, hid_lane, dw_lane);
            __syncthreads();
        }
    }

    // ---- the projection's sums ----
    v4i res[kTiles];
    int64_t m[kTiles];
    int valid[kTiles];
#pragma unroll
    for (int t = 0; t < kTiles; ++t) {
        const int p = tile_px[t] * 32 + col, row = (int)fast_div((uint32_t)p, a.pitch_o_mul, a.pitch_o_shift), ox = p - row * a.pitch_o, oc = tile_oc[t] * 32 + 16 * half;
        const bool inside = wave + kWaves * t < tiles && row < a.R && oh0 + row < a.OH && ox < a.OW;
        m[t] = (int64_t)(oh0 + row) * a.OW + ox;
        valid[t] = inside ? a.OC - oc : 0;
        res[t] = v4i{0, 0, 0, 0};
        // (an aligned chunk that holds one byte of the tensor can be read whole)
        if (a.res.r && valid[t] > 0) res[t] = *reinterpret_cast<const v4i*>(a.res.r + ((int64_t)n * a.OH * a.OW + m[t]) * a.res.r_px_stride + oc);
    }
#pragma unroll
    for (int t = 0; t < kTiles; ++t) {
        if (wave + kWaves * t >= tiles) break;
        const int oc = tile_oc[t] * 32 + 16 * half;
        float pre[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) pre[r] = (float)(acc[t][r] + s_add[oc + r]) * s_scale[oc + r];
        prefloor(pre, in_vector_registers(a.q3));
        uint32_t word[4];
        floor_sat_u8x16(pre, word);
        v4i val = {(int)word[0], (int)word[1], (int)word[2], (int)word[3]};
        if (a.res.r) {
            if (a.res.affine == 1) val = affine_residual16<false>(val, res[t], a.res);
            else if (a.res.affine == 2) val = affine_residual16<true>(val, res[t], a.res);
            else val = add_residual16_any(val, res[t], a.res);
        }
        val ^= (int)a.y_flip;
        char* dst = a.y + (int64_t)n * a.y_n + m[t] * a.y_px + oc;
        if (valid[t] >= 16) *reinterpret_cast<v4i*>(dst) = val;
        else if (valid[t] > 0) store_first(dst, val, valid[t]);
    }
}

// A work-group per (row tile, K tile); the tables by the first K tile's.
__global__ __launch_bounds__(64) void pack_inverted_point_kernel(const int8_t* w, int64_t s_row, int64_t s_k, const float* scale, int64_t s_scale, int scales, const int32_t* bias,
                                                                 int64_t s_bias, int rows, int K, int projection, char* fragments, int32_t* table) {
    const int lane = threadIdx.x, tile = (int)blockIdx.y, k_tile = (int)blockIdx.x, k_tiles = (int)gridDim.x;
    const int row = tile * 32 + (projection ? pixel_of(lane & 31) : lane & 31);
    v4i v = {0, 0, 0, 0};
    for (int i = 0; i < 16; ++i) {
        const int k = k_tile * 32 + (lane >> 5) * 16 + i;
        if (row < rows && k < K) v[i / 4] |= (int)((uint32_t)(uint8_t)w[row * s_row + k * s_k] << (8 * (i % 4)));
    }
    *reinterpret_cast<v4i*>(fragments + ((int64_t)(tile * k_tiles + k_tile) * 64 + lane) * 16) = v;
    if (k_tile != 0 || lane >= 32) return;
    const int r = tile * 32 + lane;
    int32_t sum = 0;
    if (r < rows)
        for (int k = 0; k < K; ++k) sum += w[r * s_row + k * s_k];
    const float f = r < rows ? *reinterpret_cast<const float*>(reinterpret_cast<const char*>(scale) + (scales > 1 ? r : 0) * s_scale) : 0.f;
    table[r * 4] = __float_as_int(f);
    table[r * 4 + 1] = bias && r < rows ? *reinterpret_cast<const int32_t*>(reinterpret_cast<const char*>(bias) + r * s_bias) : 0;
    table[r * 4 + 2] = sum;
    table[r * 4 + 3] = 0;
}

__global__ __launch_bounds__(64) void pack_inverted_depthwise_kernel(const int8_t* w, int64_t s_c, int64_t s_h, int64_t s_w, const float* scale, int64_t s_scale, int scales, const int32_t* bias,
                                                                     int64_t s_bias, int channels, int32_t* table) {
    const int c = (int)blockIdx.x * 64 + threadIdx.x;
    int32_t sum = 0;
    for (int i = 0; i < 3; ++i) {
        uint32_t row = 0;
        for (int j = 0; j < 3; ++j) {
            const int8_t v = c < channels ? w[c * s_c + i * s_h + j * s_w] : (int8_t)0;
            row |= (uint32_t)(uint8_t)v << (8 * j);
            sum += v;
        }
        table[c * 8 + i] = (int32_t)row;
    }
    const float f = c < channels ? *reinterpret_cast<const float*>(reinterpret_cast<const char*>(scale) + (scales > 1 ? c : 0) * s_scale) : 0.f;
    table[c * 8 + 3] = __float_as_int(f);
    table[c * 8 + 4] = bias && c < channels ? *reinterpret_cast<const int32_t*>(reinterpret_cast<const char*>(bias) + c * s_bias) : 0;
    table[c * 8 + 5] = sum;
    table[c * 8 + 6] = table[c * 8 + 7] = 0;
}

int odd16(int bytes) {  // an odd number of 16 bytes
    return 16 * (((bytes + 15) / 16) | 1);
}

// What a work-group of R output rows needs: fills the launch's fields, returns its LDS bytes.
int lay_out(InvertedResidualArgs& a, int stride, int R, int G, int buffers) {
    a.R = R;
    a.buffers = buffers;
    a.rows = (R - 1) * stride + 3;
    a.pitch = (a.W + 1 + 3) / 4 * 4;
    a.pixels = (a.rows * a.pitch + 31) / 32 * 32;
    a.px_bytes = odd16(a.x_chunks * 16);
    a.pitch_o = (a.OW + 7) / 8 * 8;
    a.items = R * (a.pitch_o / 8);
    a.tiles_px = (R * a.pitch_o + 31) / 32;
    a.tiles_oc = (a.OC + 31) / 32;
    // (the last results of a row read up to two dwords past it)
    a.cs = odd16(16 + a.pixels + 16 * stride);
    a.cs2 = odd16(a.tiles_px * 32);
    a.intervals = (a.hid_tiles + G - 1) / G;
    a.strips = (a.OH + R - 1) / R;
    a.at_mask = a.pixels * a.px_bytes;
    a.at_hid = a.at_mask + a.pixels;
    a.at_dw = a.at_hid + buffers * G * 32 * a.cs;
    a.at_t3 = a.at_dw + buffers * G * 32 * a.cs2;
    return a.at_t3 + 32 * a.tiles_oc * 8;
}

constexpr int kLdsOfUnit = 160 * 1024;

template <int kStride, int kTiles, int kG, int kKS, int kBuffers>
int launch(const InvertedResidualArgs& a, int bytes, hipStream_t s) {
    // (more than 64 KB has to be asked for, on every device)
    if (bytes > 64 * 1024)
        CHX_HIP_CALL(hipFuncSetAttribute(reinterpret_cast<const void*>(&inverted_residual_kernel<kStride, kTiles, kG, kKS, kBuffers>), hipFuncAttributeMaxDynamicSharedMemorySize, kLdsOfUnit));
    inverted_residual_kernel<kStride, kTiles, kG, kKS, kBuffers><<<8 * a.xcd_chunk, 64 * kWaves, bytes, s>>>(a);
    return launch_check("inverted_residual_kernel");
}

template <int kTiles, int kG, int kBuffers>
int launch_steps(const InvertedResidualArgs& a, int stride, int bytes, hipStream_t s) {
    if constexpr (kBuffers == 2) {
        if (a.KS == 5) return stride == 1 ? launch<1, kTiles, kG, 5, kBuffers>(a, bytes, s) : launch<2, kTiles, kG, 5, kBuffers>(a, bytes, s);
    }
    if (stride == 1) return a.KS == 1 ? launch<1, kTiles, kG, 1, kBuffers>(a, bytes, s) : launch<1, kTiles, kG, 3, kBuffers>(a, bytes, s);
    return a.KS == 1 ? launch<2, kTiles, kG, 1, kBuffers>(a, bytes, s) : launch<2, kTiles, kG, 3, kBuffers>(a, bytes, s);
}

// The two sides of whether the block is one launch, in us, fitted to 1,059 blocks of 8 to 160 channels, expanded 1 to 6 times, to 8 to
// 320, on 1 to 128 images of 4 to 150, each measured both ways inside a recording (within 8 and 7 %).  A strip expands its halo
// again: where LDS holds a row or two of a wide image at a time, or many channels leave, that costs more than the expanded
// activations' way through memory.  us as three launches and as one: 54 x 8 -> 48 -> 80 at 86x86 46 and 83, 60 x 128 -> 768 -> 208 at 51x51
// 161 and 290, 70 x 24 -> 144 -> 104 at 104x104 155 and 340; 126 x 16 -> 48 -> 8 at 99x99 75 and 129.  All as one launch were 0.92 of
// the time of three on average, one in seven more than 5 % slower (up to 2.1 times); by this choice 0.89, nine of them, by up
// to 20 %; of 400 others, six by up to 14 %.  All blocks of a MobileNetV2 on 1 to 128 images are one launch, but for what the refusal below names.
double time_of_launches(const InvertedResidualArgs& a) {
    auto pad = [](int64_t n, int64_t by) { return (double)((n + by - 1) / by * by); };
    const int64_t channels = (int64_t)a.x_chunks * 16, hid = (int64_t)a.hid_tiles * 32;
    const double in = 1e-6 * (double)a.N * a.H * a.W, out = 1e-6 * (double)a.N * a.OH * a.OW, h = (double)hid, oc = pad(a.OC, 16);
    const double expansion = std::max(2.4e-3 * in * pad(channels, 64) * pad(hid, 64), 0.28 * in * h), projection = std::max(2.4e-3 * out * pad(hid, 64) * pad(a.OC, 64), 0.28 * out * oc);
    return 11.6 + expansion + projection + in * (3.8 + 0.104 * h) + 0.50 * out * h;
}

double time_of_block(const InvertedResidualArgs& a, int64_t blocks) {
    auto shares = [](int n, int by) { return (double)((n + by - 1) / by); };
    const int per = kWaves / a.G, tiles = a.tiles_px * a.tiles_oc;
    const double runs = shares(a.pixels / 32, per), items = shares((a.items + 1) / 2, per), mine = shares(tiles, kWaves), rows = (double)a.rows * a.W * a.x_chunks / 512.0;
    const bool two = 2 * a.lds <= kLdsOfUnit && tiles <= kWaves && a.G <= 2 && blocks > 256;
    const double rounds = two ? 1.2 * (blocks > 2048 ? blocks / 512.0 : (double)((blocks + 511) / 512)) : (double)((blocks + 255) / 256);
    const double filled = 2.05 + 1e-3 * rounds * ((a.intervals + 2) * (944.0 + runs * (109.0 + 46.0 * a.KS) + 300.0 * items + 54.0 * mine * a.G) + 23.0 * rows + 92.0 * (mine + 1));
    if (blocks > 256) return filled;
    // one round: the start is most of it
    const double start = 6.7 + 1e-3 * ((a.intervals + 2) * (76.0 + 58.0 * runs * a.KS + 349.0 * items) + 348.0 * (mine + 1));
    return start > 13.0 && filled > start ? 0.65 * start + 0.35 * filled : start;
}

}  // namespace

int plan_inverted_residual(InvertedResidualArgs* launch, int stride) {
    InvertedResidualArgs& a = *launch;
    // Rows per strip, and tiles of channels per interval.  A strip expands the rows of its halo again, so few rows cost work;
    // many leave compute units idle, or LDS for one work-group only; many channels per interval mean few barriers, each
    // wavefront on channels of its own, and little left to share out where the strip is large.  The least of rounds x
    // instructions of the busiest wavefront, with constants fitted to measured choices for the eleven blocks of a MobileNetV2
    // (7x7 to 112x112) on 1 to 128 images.  Three of them are more than 5 % from their best choice: 64 -> 384 -> 64 at 14x14 x
    // 128 (18.0 us, 15.5 the best), 32 -> 192 -> 32 x 32 (11.9, 10.7) and 24 -> 144 -> 32 x 32 (13.5, 12.6).
    //
    // More than 256 channels out are two or three tiles for a wavefront, whose filters every strip reads for itself, and the
    // projection's own launch has its channels spread over the chip: 160 -> 960 -> 320 at 7x7 takes, as three launches and as
    // one, 14.1 and 16.9 us on 1 image, 15.6 and 19.2 on 32, 19.0 and 19.2 on 64 (448 rows), 28.5 and 23.7 on 128 (896 rows).
    if ((a.OC + 31) / 32 > kWaves && (int64_t)a.N * a.OH < 512) CHX_FAIL(CHX_HIP_EUNSUPPORTED, "inverted residual: too few rows for so many channels");
    //
    // With one buffer of each kind (the kernel's kBuffers) LDS holds about twice the rows: 16 -> 96 -> 24 at 112x112 takes four per strip
    // for two, and expands nine rows where it expanded ten; the price is a second barrier per interval.  In us with two and with one, 128
    // images: 77.5 and 63.2 (16 -> 96 -> 24 at 112x112), 68.1 and 63.1 (24 -> 144 -> 24 at 56x56), 23.7 and 21.4 (32 -> 192 -> 32 at 28x28);
    // 64 images 48.9 and 37.5, 39.1 and 33.6, 15.5 and 15.2; 14x14 and 7x7, where a strip is most of an image anyway, 18.4
    // and 19.0.  The constants are those of 182 blocks on 1 to 128 images, each with all rows and tiles measured: of 31 that take one
    // buffer none was slower, the most 0.60 of the time.  Where one round does not fill the chip a second barrier is all it is.
    // (160 input channels, and two tiles of the projection with other than 16 or 32 input channels, do not fit the registers.)
    int best = 0, best_g = 1, best_buffers = 2, rows_of_two = 0, tiles_of_two = 1;
    double least = 0;
    for (int buffers = 2; buffers >= 1; --buffers) {
        for (int G = 1; G <= (buffers == 1 ? 2 : 8); G *= 2) {
            if (G > 1 && G / 2 >= a.hid_tiles) break;
            for (int R = 1; R <= a.OH && R <= 16; ++R) {
                const int bytes = lay_out(a, stride, R, G, buffers), tiles = a.tiles_px * a.tiles_oc;
                const int64_t blocks = (int64_t)a.strips * a.N;
                if (bytes > kLdsOfUnit || tiles > kMostTiles * kWaves || (G == 8 && tiles > 2 * kWaves)) continue;
                if (buffers == 1 && (blocks <= 256 || a.KS == 5 || tiles > (G == 1 && a.KS == 1 ? 2 : 1) * kWaves)) continue;
                const int per = kWaves / G;  // wavefronts that share the runs and items of a tile of channels
                auto shares = [](int n, int by) { return (double)((n + by - 1) / by); };
                const double interval = shares(a.pixels / 32, per) * (120.0 + 14.0 * a.KS) + shares((a.items + 1) / 2, per) * 132.0 + shares(tiles, kWaves) * 13.0 * G + (buffers == 2 ? 190.0 : 300.0);
                const double work = (a.intervals + (buffers == 2 ? 2.0 : 0.5)) * interval + (buffers == 2 ? 850.0 : 1300.0) + a.rows * a.W * a.x_chunks / 512 * 25.0;
                const bool two = 2 * bytes <= kLdsOfUnit && (buffers == 1 || (tiles <= kWaves && G <= 2)) && blocks > 256;  // work-groups on a compute unit at once
                const double cost = two ? (blocks > 2048 ? blocks / 512.0 : (double)((blocks + 511) / 512)) * (buffers == 2 ? 1.232 : 1.3) * work : (double)((blocks + 255) / 256) * work;
                if (best == 0 || cost < least) {
                    least = cost;
                    best = R;
                    best_g = G;
                    best_buffers = buffers;
                }
            }
        }
        if (buffers == 2) {
            rows_of_two = best;
            tiles_of_two = best_g;
        }
    }
    if (best == 0) CHX_FAIL(CHX_HIP_EUNSUPPORTED, "inverted residual: a row does not fit");
    // (the estimate for one buffer is within 14 %: what two would be refused for has to be that much better)
    double here = best_buffers == 1 ? 1.15 * (0.7 + 2.35e-3 * least) : 0.0;
    if (rows_of_two != 0) {
        a.G = tiles_of_two;
        a.lds = lay_out(a, stride, rows_of_two, tiles_of_two, 2);
        const double two = time_of_block(a, (int64_t)a.strips * a.N);
        here = best_buffers == 1 ? std::min(here, two) : two;
    }
    const double launches = time_of_launches(a);  // (up to 16 us most of it is that they are three)
    if (here > (launches < 16.0 ? launches + 2.3 : 0.93 * launches + 1.0)) CHX_FAIL(CHX_HIP_EUNSUPPORTED, "inverted residual: slower than its convolutions");
    a.G = best_g;
    a.lds = lay_out(a, stride, best, best_g, best_buffers);
    const int64_t blocks = (int64_t)a.strips * a.N;
    if (blocks >= (int64_t(1) << 28)) CHX_FAIL(CHX_HIP_EUNSUPPORTED, "inverted residual: 2^28 strips or more");
    a.blocks = (int32_t)blocks;
    a.xcd_chunk = (int32_t)((blocks + 7) / 8);
    magic_divisor((uint32_t)a.strips, &a.strips_mul, &a.strips_shift);
    magic_divisor((uint32_t)a.pitch, &a.pitch_mul, &a.pitch_shift);
    magic_divisor((uint32_t)a.pitch_o, &a.pitch_o_mul, &a.pitch_o_shift);
    magic_divisor((uint32_t)(a.W * a.x_chunks), &a.row_mul, &a.row_shift);
    magic_divisor((uint32_t)a.x_chunks, &a.chunks_mul, &a.chunks_shift);
    magic_divisor((uint32_t)a.tiles_oc, &a.oct_mul, &a.oct_shift);
    magic_divisor((uint32_t)(a.pitch_o / 8), &a.blk_mul, &a.blk_shift);
    return CHX_HIP_OK;
}

int launch_inverted_residual(const InvertedResidualArgs& a, int stride, hipStream_t s) {
    const int bytes = a.lds, per_wave = (a.tiles_px * a.tiles_oc + kWaves - 1) / kWaves;
    if (a.buffers == 1) {
        if (per_wave == 2) return stride == 1 ? launch<1, 2, 1, 1, 1>(a, bytes, s) : launch<2, 2, 1, 1, 1>(a, bytes, s);
        return a.G == 1 ? launch_steps<1, 1, 1>(a, stride, bytes, s) : launch_steps<1, 2, 1>(a, stride, bytes, s);
    }
    if (per_wave == 1) {
        switch (a.G) {
            case 1: return launch_steps<1, 1, 2>(a, stride, bytes, s);
            case 2: return launch_steps<1, 2, 2>(a, stride, bytes, s);
            case 4: return launch_steps<1, 4, 2>(a, stride, bytes, s);
            default: return launch_steps<1, 8, 2>(a, stride, bytes, s);
        }
    }
    switch (a.G) {
        case 1: return launch_steps<kMostTiles, 1, 2>(a, stride, bytes, s);
        case 2: return launch_steps<kMostTiles, 2, 2>(a, stride, bytes, s);
        case 4: return launch_steps<kMostTiles, 4, 2>(a, stride, bytes, s);
        default: return launch_steps<2, 8, 2>(a, stride, bytes, s);  // (the filters of three tiles do not fit the registers)
    }
}

int pack_inverted_point(const chx_hip_tensor& w, const chx_hip_tensor& scale, const chx_hip_tensor* bias, bool projection, int row_tiles, int k_tiles,
                        char* fragments, int32_t* table, hipStream_t s) {
    pack_inverted_point_kernel<<<dim3((unsigned)k_tiles, (unsigned)row_tiles), 64, 0, s>>>(
            static_cast<const int8_t*>(w.data), w.strides[0], w.strides[1], static_cast<const float*>(scale.data), scale.ndim ? scale.strides[0] : 0, (int)numel(scale),
            bias ? static_cast<const int32_t*>(bias->data) : nullptr, bias ? bias->strides[0] : 0, (int)w.shape[0], (int)w.shape[1], projection ? 1 : 0, fragments, table);
    return launch_check("pack_inverted_point_kernel");
}

int pack_inverted_depthwise(const chx_hip_tensor& w, const chx_hip_tensor& scale, const chx_hip_tensor* bias, int tiles, int32_t* table, hipStream_t s) {
    pack_inverted_depthwise_kernel<<<(unsigned)((tiles * 32 + 63) / 64), 64, 0, s>>>(
            static_cast<const int8_t*>(w.data), w.strides[0], w.strides[2], w.strides[3], static_cast<const float*>(scale.data), scale.ndim ? scale.strides[0] : 0, (int)numel(scale),
            bias ? static_cast<const int32_t*>(bias->data) : nullptr, bias ? bias->strides[0] : 0, (int)w.shape[0], table);
    return launch_check("pack_inverted_depthwise_kernel");
}

}  // namespace chx
