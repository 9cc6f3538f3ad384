// The packed-weight convolution for 3x3 filters over an image whose results have its size: pixels from LDS, weights straight
// into registers.
//
// conv_mfma_kernel brings a tile's pixels into LDS once per filter tap, nine times what the tile covers, and its weights beside
// them.  Here a work-group brings the one run of pixels that all taps of its 64 or 128 pixels fall on (conv_split_kernel's patch,
// pixels an odd number of 16 bytes apart, taps outside the image read zero points), once, and a wavefront has 32 channels of its
// own, whose weights it reads from memory in the order of the fragments, several steps ahead: one barrier per tile.
// us inside a recording, the faster of the staged and the small tiles, and this kernel's faster tile: 128 -> 128 channels of
// 28x28, 32 images 10.8 and 8.6, 8 images 7.5 and 4.9, 64 images 15.0 and 13.3; 512 -> 512 of 7x7, 64 images 20.4 and 13.3; 64 -> 64 of 56x56, 64 images
// 20.5 and 15.3, 8 images 7.4 and 5.2; 256 -> 256 of 14x14, 64 images 15.9 and 12.1, 8 images 5.9 and 6.0; 144 -> 328 of 21x21, 22
// images 16.0 and 11.3; 128 -> 368 of 29x29, 48 images 27.9 and 28.3.  So it is measured per shape beside them (tune_conv_mfma).
// A wavefront's step of 32 K bytes is one fragment from memory, two from LDS and two products: at the matrix cores' full rate that is 64 bytes
// a cycle from L2 and 128 from LDS for a compute unit, all that there is of either, and about 60 % of it is reached.
#include <type_traits>

#include "conv_mfma.h"
#include "conv_device.h"

namespace chx {
namespace {

struct ConvSameArgs {
    ConvMfmaArgs conv;
    uint32_t x_flip;
    int32_t tiles_per_xcd, patch_chunks, patch_pitch, segments;  // of a filter: (tap, kU steps)
    uint32_t tiles_px_mul, tiles_px_shift, chunks_mul, chunks_shift;
};

// kU: steps of 32 K bytes in a segment; kT: segments of an iteration, whose weights are requested one iteration ahead.  kXT: tiles of
// 32 pixels of a wavefront; kWO, kWP: wavefronts along the channels and along the pixels.
template <int kU, int kT, int kXT, int kWO, int kWP>
__global__ __launch_bounds__(64 * kWO * kWP, 2) void conv_same_kernel(ConvSameArgs) {
    constexpr int kThreads = 64 * kWO * kWP, kPx = 32 * kXT * kWP, kRing = kU * kT;
    constexpr int kAhead = kU < 4 ? kU : 3, kRows = kU < 4 ? kAhead + 1 : kRing % 4 == 0 ? 4 : 6;  // steps that the pixels are read ahead; their registers
    static_assert(kAhead < kRows && kRing % kRows == 0 && kAhead <= kU, "");
    __shared__ __attribute__((aligned(16))) float s_scale[32 * kWO], s_bias[32 * kWO];
    __shared__ __attribute__((aligned(16))) int32_t s_add[32 * kWO];
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const ConvSameArgs& args = kernel_arguments<ConvSameArgs>();
    const ConvMfmaArgs& a = args.conv;
    const int idx = (int)(blockIdx.x >> 3), tile = (int)(blockIdx.x & 7) * args.tiles_per_xcd + idx;
    if (idx >= args.tiles_per_xcd || tile >= a.tiles_oc * a.tiles_px) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, half = lane >> 5, wo = wave % kWO, wp = wave / kWO;
    // an XCD's run of tiles: all pixels of a few channel tiles, so that their weights are fetched into one L2
    const int oc_tile = (int)fast_div((uint32_t)tile, args.tiles_px_mul, args.tiles_px_shift), px_tile = tile - oc_tile * a.tiles_px;
    const int oc0 = oc_tile * 32 * kWO, m0 = px_tile * kPx, last_px = (int)a.M - 1;

    // fragments of 32 channels are 1 KB of wf (fragment_offset in conv_mfma.hip), whose rows a lane takes in its own order
    const int row = channel_of(col);
    const uint32_t w_lane = (uint32_t)((row >> 4) * 512 + half * 256 + (row & 15) * 16);
    const char* const w = reinterpret_cast<const char*>(a.wf) + (int64_t)min(oc0 / 32 + wo, (a.OC - 1) >> 5) * 32 * a.KP;
    auto fragment = [&](int step) { return *reinterpret_cast<const v4i*>(w + (uint32_t)step * 1024u + w_lane); };
    v4i ring[kRing];
    {
        constexpr int kBatch = 4;
        const int first = m0 - a.W - 1, total = args.patch_chunks, per_px = a.C16 >> 4;
        const bool inside = first >= 0 && first + kPx + 2 * a.W + 2 <= (int)a.M;
        const char* const from = a.x + (int64_t)first * a.x_w_stride;
        v4i v[kBatch];
        int to[kBatch];
        auto load = [&](int i0) {
#pragma unroll
            for (int b = 0; b < kBatch; ++b) {
                const int i = min(i0 + b * kThreads, total - 1), px = (int)fast_div((uint32_t)i, args.chunks_mul, args.chunks_shift), c = i - px * per_px;
                to[b] = px * args.patch_pitch + c * 16;
                if (inside) v[b] = *reinterpret_cast<const v4i*>(from + ((uint32_t)px * (uint32_t)a.x_w_stride + (uint32_t)c * 16u));
                else v[b] = *reinterpret_cast<const v4i*>(a.x + ((uint32_t)min(max(first + px, 0), last_px) * (uint32_t)a.x_w_stride + (uint32_t)c * 16u));
            }
        };
        load(tid);
#pragma unroll
        for (int i = 0; i < kRing; ++i) ring[i] = fragment(i);
        if (tid < 32 * kWO) {
            const int ch = min(oc0 + tid, a.OC - 1);
            const int32_t bias = a.bias ? a.bias[ch] : 0;
            s_scale[tid] = a.rq.x_scale * (a.w_scale_len > 1 ? a.w_scale[ch] : a.w_scale[0]);
            s_add[tid] = a.corr_mult * a.wsum[ch] + (a.rq.bias_mode == kBiasOnnxInt32 ? bias : 0);
            s_bias[tid] = a.rq.bias_mode == kBiasReferenceFloat ? (float)bias : 0.f;
        }
        if (tid < kU * 2) {
            const int fill = (int)((uint32_t)(a.x_zp & 0xff) * 0x01010101u ^ args.x_flip);
            *reinterpret_cast<v4i*>(lds + tid * 16) = v4i{fill, fill, fill, fill};
        }
        for (int i0 = tid; i0 < total; i0 += kBatch * kThreads) {
            if (i0 != tid) load(i0);
#pragma unroll
            for (int b = 0; b < kBatch; ++b) *reinterpret_cast<v4i*>(lds + kU * 32 + to[b]) = v[b] ^ (int)args.x_flip;
        }
    }
    int x_off[kXT];
    uint32_t taps[kXT];
#pragma unroll
    for (int j = 0; j < kXT; ++j) {
        const int p = (wp * kXT + j) * 32 + col;
        const uint32_t m = (uint32_t)min(m0 + p, last_px), r = fast_div(m, a.ow_mul, a.ow_shift), ow = m - r * (uint32_t)a.W;
        const uint32_t n = fast_div(r, a.oh_mul, a.oh_shift), oh = r - n * (uint32_t)a.H;
        const uint32_t cols = (ow > 0 ? 1u : 0u) | 2u | ((int)ow < a.W - 1 ? 4u : 0u);
        taps[j] = (oh > 0 ? cols : 0u) | cols << 3 | ((int)oh < a.H - 1 ? cols << 6 : 0u);
        x_off[j] = kU * 32 + p * args.patch_pitch + 16 * half;
    }
    lds_barrier();

    // (in the order that it is written in: see bottleneck_kernel)
    v16i acc[kXT];
#pragma unroll
    for (int j = 0; j < kXT; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const v4i v = *reinterpret_cast<const v4i*>(s_add + wo * 32 + 16 * half + 4 * i);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[j][4 * i + e] = v[e];
        }
    {
        int tap = 0, tap_off = 0, kw = 0, k_in = 0, off[kXT], off_next[kXT];
        int column = args.patch_pitch, to_row = (a.W - 2) * args.patch_pitch, k_end = a.C64;
        keep_scalar(column);
        keep_scalar(to_row);
        keep_scalar(k_end);
        auto offsets = [&](int (&to)[kXT]) {  // of the segment, and on to the next (behind the last: zero points)
#pragma unroll
            for (int j = 0; j < kXT; ++j) to[j] = (taps[j] >> tap) & 1 ? x_off[j] + tap_off + k_in : 16 * half;
            k_in += kU * 32;
            const bool next_tap = k_in == k_end, next_row = next_tap && kw == 2;
            k_in = next_tap ? 0 : k_in;
            tap += next_tap ? 1 : 0;
            tap_off += next_row ? to_row : next_tap ? column : 0;
            kw = next_row ? 0 : next_tap ? kw + 1 : kw;
        };
        v4i px[kRows][kXT];
        auto read = [&](v4i (&to)[kXT], const int (&from)[kXT], int k) {
#pragma unroll
            for (int j = 0; j < kXT; ++j) to[j] = *reinterpret_cast<const v4i*>(lds + from[j] + k * 32);
        };
        offsets(off);
#pragma unroll
        for (int k = 0; k < kAhead; ++k) read(px[k], off, k);
        auto iteration = [&](auto last, int done) {
            const int ahead = done * kU + kRing;
#pragma unroll
            for (int t = 0; t < kT; ++t) {
                offsets(off_next);
#pragma unroll
                for (int k = 0; k < kU; ++k) {
                    const int i = t * kU + k;
                    if (k + kAhead < kU) read(px[(i + kAhead) % kRows], off, k + kAhead);
                    else read(px[(i + kAhead) % kRows], off_next, k + kAhead - kU);
#pragma unroll
                    for (int j = 0; j < kXT; ++j) acc[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(ring[i], px[i % kRows][j], acc[j], 0, 0, 0);
                    if constexpr (!decltype(last)::value) ring[i] = fragment(ahead + i);
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int j = 0; j < kXT; ++j) off[j] = off_next[j];
            }
        };
        const int segments = args.segments;
#pragma unroll 1
        for (int done = 0; done < segments - kT; done += kT) iteration(std::false_type(), done);
        iteration(std::true_type(), segments - kT);
    }

    const QuantProduct q = in_vector_registers(a.qp);
    const bool biased = a.rq.bias_mode == kBiasReferenceFloat;
    const int oc = oc0 + wo * 32 + 16 * half;
#pragma unroll
    for (int j = 0; j < kXT; ++j) {
        const int m = m0 + (wp * kXT + j) * 32 + col;
        float pre[16];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const v4f s = *reinterpret_cast<const v4f*>(s_scale + wo * 32 + 16 * half + 4 * i);
#pragma unroll
            for (int e = 0; e < 4; ++e) pre[4 * i + e] = (float)acc[j][4 * i + e] * s[e];
        }
        if (biased) {
#pragma unroll
            for (int e = 0; e < 16; ++e) pre[e] = pre[e] + s_bias[wo * 32 + 16 * half + e];
        }
        if (q.path == 3) {  // (the path is the same in every lane)
#pragma unroll
            for (int e = 0; e < 16; ++e) pre[e] = quantize_prefloor_u8<3>(pre[e], q);
        } else if (q.path == 2) {
#pragma unroll
            for (int e = 0; e < 16; ++e) pre[e] = quantize_prefloor_u8<2>(pre[e], q);
        } else {
#pragma unroll
            for (int e = 0; e < 16; ++e) pre[e] = quantize_prefloor_u8<1>(pre[e], q);
        }
        uint32_t word[4];
        floor_sat_u8x16(pre, word);
        const v4i codes = v4i{(int)word[0], (int)word[1], (int)word[2], (int)word[3]} ^ (int)a.y_flip;
        if (m > last_px || oc >= a.OC) continue;
        char* const dst = a.y + (int64_t)m * a.y_px_stride + oc;
        if (oc + 16 <= a.OC) *reinterpret_cast<v4i_u*>(dst) = codes;
        else
            for (int e = 0; e < a.OC - oc; ++e) dst[e] = (char)((uint32_t)codes[e / 4] >> (8 * (e % 4)));
    }
}

constexpr int kLdsOfUnit = 160 * 1024, kTableBytes = 3 * 4 * 256;

int pitch_of(const ConvMfmaArgs& a) {
    return a.C16 % 32 == 0 ? a.C16 + 16 : a.C16;
}

int bytes_of(const ConvMfmaArgs& a, int tile_px) {  // (a pixel's channels are read up to C64)
    return 256 + (tile_px + 2 * a.W + 2) * pitch_of(a) + 64;
}

template <int kU, int kT, int kXT, int kWO, int kWP>
int launch(const ConvMfmaArgs& a, uint32_t flip, hipStream_t s) {
    const int px = 32 * kXT * kWP, bytes = bytes_of(a, px);
    ConvSameArgs args;
    args.conv = a;
    args.x_flip = flip;
    args.tiles_per_xcd = (int)(((int64_t)a.tiles_oc * a.tiles_px + 7) / 8);
    args.patch_pitch = pitch_of(a);
    args.patch_chunks = (px + 2 * a.W + 2) * (a.C16 / 16);
    args.segments = 9 * (a.C64 / 32) / kU;
    magic_divisor((uint32_t)a.tiles_px, &args.tiles_px_mul, &args.tiles_px_shift);
    magic_divisor((uint32_t)(a.C16 / 16), &args.chunks_mul, &args.chunks_shift);
    if (bytes > 60 * 1024)  // (has to be asked for, on every device)
        CHX_HIP_CALL(hipFuncSetAttribute(reinterpret_cast<const void*>(&conv_same_kernel<kU, kT, kXT, kWO, kWP>), hipFuncAttributeMaxDynamicSharedMemorySize, kLdsOfUnit - kTableBytes));
    conv_same_kernel<kU, kT, kXT, kWO, kWP><<<8 * args.tiles_per_xcd, 64 * kWO * kWP, bytes, s>>>(args);
    return launch_check("conv_same_kernel");
}

// Steps of a segment for the K steps of a tap: 0 where there is no kernel.
int segment_of(int steps) {
    return steps == 2 || steps == 4 ? steps : steps % 8 == 0 ? 8 : steps % 6 == 0 ? 6 : 0;
}

template <int kXT, int kWO, int kWP>
int launch_steps(const ConvMfmaArgs& a, uint32_t flip, hipStream_t s) {
    switch (segment_of(a.C64 / 32)) {
        case 2: return launch<2, 3, kXT, kWO, kWP>(a, flip, s);
        case 4: return launch<4, 3, kXT, kWO, kWP>(a, flip, s);
        case 6: return launch<6, 1, kXT, kWO, kWP>(a, flip, s);
        default: return launch<8, 1, kXT, kWO, kWP>(a, flip, s);
    }
}

}  // namespace

bool conv_same_has(int tile_oc, int tile_px, int waves) {
    for (const ConvSplitTile& t : kConvSameTiles)
        if (t.oc == tile_oc && t.px == tile_px && t.waves == waves) return true;
    return false;
}

bool conv_same_takes(const ConvMfmaArgs& a, int tile_px) {
    return a.wf != nullptr && a.KH == 3 && a.KW == 3 && a.ph == 1 && a.pw == 1 && a.sh == 1 && a.sw == 1 && a.OH == a.H && a.OW == a.W && a.qp.path != 0 && !a.res.r && a.oc_split == 0 &&
           segment_of(a.C64 / 32) != 0 && a.x_h_stride == (int64_t)a.W * a.x_w_stride && (a.x_n_stride == (int64_t)a.H * a.x_h_stride || a.M == (int64_t)a.OH * a.OW) &&
           a.W < 8192 && a.C16 <= 4096 && a.M < (int64_t(1) << 30) && (int64_t)(tile_px + 2 * a.W + 2) * pitch_of(a) + 512 <= kLdsOfUnit - kTableBytes;
}

int launch_conv_same(const ConvMfmaArgs& a, int tile_oc, int tile_px, int waves, bool x_unsigned, hipStream_t s) {
    const uint32_t flip = x_unsigned ? 0x80808080u : 0u;
#define CHX_SAME(XT, WO, WP) \
    if (tile_oc == 32 * WO && tile_px == 32 * XT * WP && waves == WO * WP) return launch_steps<XT, WO, WP>(a, flip, s);
    CHX_SAME(1, 2, 2)
    CHX_SAME(2, 2, 2)
    CHX_SAME(2, 4, 1)
    CHX_SAME(2, 4, 2)
#undef CHX_SAME
    CHX_FAIL(CHX_HIP_EINVAL, "conv_same: no kernel for a %dx%d tile with %d wavefronts", tile_oc, tile_px, waves);
}

}  // namespace chx
