// The packed-weight convolution for launches with few output tiles: small tiles whose K is shared out over the
// wavefronts of a work-group.
//
// With one image (or a few) the tiles of conv_mfma_kernel occupy a fraction of the 256 compute units, each walking a K of
// up to 4608 bytes through LDS stage by stage: 7 to 14 us per layer of ResNet-50 whatever the layer's size.  Here a
// work-group owns R output channels x R*PN pixels (R = 16 or 32), and its W wavefronts take K apart: fragments come
// straight from memory (16 bytes per lane: the packed weights and channels-last pixels have them contiguous), several
// steps in flight, no barrier until the W partial sums meet in LDS.  Weights are read once per pixel tile and pixels once
// per channel tile, from L2, so this is for launches bound by latency; which configuration runs is measured per shape
// (tune_conv_mfma).  ResNet-50 on one image, all 55 launches replayed: 370 us with the staged tiles alone, 308 with these.
// The weights have a layout of their own (ConvMfmaArgs::wf), in which a step's fragment is in one or two places: from the staged
// tiles' one ResNet-50 takes 258 us on one image and 372 on eight, from this 240 and 360.
//
// Arguments, requantization, residual sums, pairs and storage are those of conv_mfma_kernel; filter taps outside the
// image are replaced by the zero point on the fragment.
//
// With several taps a tile's pixels are gathered once per tap, 32 or 64 bytes from a pixel at a time: nine times 32 x 256
// bytes for what lies in 62 x 256.  Where the results have the image's own size those taps fall on one run of pixels of the
// dense image, and kPatch brings that run into LDS, once, while the weights of up to nine steps are on their way; a step then
// is weights from memory and a 16-byte LDS read per lane, pixels an odd number of 16 bytes apart, taps
// outside the image read 64 bytes of zero point.  In us, best tile with the pixels from memory and from LDS, launches
// back to back with weights of their own, 3x3 filters: one image, 512 channels at 7x7 8.5 and 5.9, 256 at 14x14 5.4 and 4.6,
// 128 at 28x28 4.8 and 4.3, 64 at 56x56 3.9 and 4.4; eight images, 11.9 and 7.9, 9.8 and 6.8, 7.1 (staged tiles) and 8.2,
// 6.9 (staged tiles) and 8.9.  So both are measured per shape.
#include <type_traits>

#include "conv_mfma.h"
#include "conv_device.h"

namespace chx {
namespace {

// Four codes of the convolution and four of the residual -> four codes of the sum (affine_residual16).
__device__ __forceinline__ uint32_t affine_residual4(uint32_t c, uint32_t r, const ResidualAdd& p) {
    const uint32_t cw = c ^ p.c_flip, rw = r ^ p.r_flip;
    float t[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        t[e] = __builtin_fmaf((float)((rw >> (8 * e)) & 0xffu), p.kr, p.k0);
        t[e] = __builtin_fmaf((float)((cw >> (8 * e)) & 0xffu), p.kc, t[e]);
        if (p.affine == 2) t[e] = __builtin_fmaxf(t[e], p.floor_pre);
    }
    return floor_sat_u8x4(t[0], t[1], t[2], t[3]);
}

typedef float v4f_u __attribute__((ext_vector_type(4), aligned(4)));

struct ConvSplitArgs {
    ConvMfmaArgs conv;
    uint32_t x_flip;
    int32_t rne, tiles_per_xcd;
    uint32_t tiles_px_mul, tiles_px_shift, c64_mul, c64_shift, kw_mul, kw_shift;  // magic_divisor(tiles_px), (C64), (KW): a division costs some 150 cycles
    int32_t patch_chunks, patch_pitch;       // kPatch: 16-byte chunks of the patch, bytes from a pixel to the next in LDS
    uint32_t chunks_mul, chunks_shift;       // magic_divisor(chunks per pixel)
};

// Where the pixels come from: one filter tap, from memory; several taps, from memory; several taps over an image whose
// results have its own size, from LDS.
enum Form { kPoint, kTaps, kPatch };

// (two wavefronts per SIMD promised, so that the sums stay out of the accumulation registers: see conv_stem_kernel)
template <int R, int PN, int W, Form kForm, int kDepth>
__global__ __launch_bounds__(64 * W, 2) void conv_split_kernel(ConvSplitArgs) {
    constexpr int kGroups = 64 / R, kStep = 16 * kGroups;  // K bytes per MFMA: 32 or 64
    constexpr int kQuads = R * R / 256;                    // groups of four result registers: 4 or 1
    constexpr int kUnits = PN * kQuads;
    using acc_t = typename std::conditional<R == 32, v16i, v4i>::type;
    __shared__ __attribute__((aligned(16))) v4i part[W > 1 ? W : 1][W > 1 ? kUnits : 1][64];
    extern __shared__ __attribute__((aligned(16))) char patch[];  // kPatch: 64 bytes of the zero point, then the pixels

    const ConvSplitArgs args = kernel_arguments<ConvSplitArgs>();
    const ConvMfmaArgs& a = args.conv;
    const int idx = (int)(blockIdx.x >> 3), tile = (int)(blockIdx.x & 7) * args.tiles_per_xcd + idx;
    if (idx >= args.tiles_per_xcd || tile >= a.tiles_oc * a.tiles_px) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane % R, group = lane / R;
    // an XCD's run of tiles: all pixels of a few channel tiles, so that their weights are fetched into one L2
    const int oc_tile = (int)fast_div((uint32_t)tile, args.tiles_px_mul, args.tiles_px_shift), px_tile = tile - oc_tile * a.tiles_px;
    const int oc0 = oc_tile * R, oc = oc0 + col;

    // Every kernel of a network starts with cold caches (what the previous one wrote has to become visible to all XCDs),
    // so a round trip to memory costs more than a microsecond here and the kernel is a chain of them.  The weights of the
    // first steps are requested before the pixels' addresses are known, and the operands of the epilogue before the loop.
    struct Step {
        v4i w, x[kForm == kPatch ? 1 : PN];
    };
    const int steps = a.KP / kStep, per = (steps + W - 1) / W, lo = wave * per, hi = min(steps, lo + per), last = hi - 1;
    // (a fragment in one or two places: 8 lines of 128 bytes for a load of 1 KB; in the staged tiles' layout it is 16 or 32)
    const uint32_t w_off = (uint32_t)(oc >> 5) * (uint32_t)(32 * a.KP) + (uint32_t)((oc & 31) >> 4 << 9) + (uint32_t)((group >> 1 << 10) + ((group & 1) << 8) + (oc & 15) * 16);
    auto load_w = [&](int step, Step& s) {
        // (past the wavefront's last step: that step again, see gemm_i8.hip)
        const uint32_t k = (uint32_t)(min(step, last) * kStep);
        s.w = *reinterpret_cast<const v4i*>(a.wf + (k * 32 + w_off));
    };
    const int fill = (int)((uint32_t)(a.x_zp & 0xff) * 0x01010101u);
    // The patch: the pixels that the taps of the tile's pixels fall on are one run of the dense image.  (Pixels outside x are
    // replaced by others: only taps outside the image look at them.)
    constexpr int kBatch = W >= 8 ? 4 : 8, kThreads = 64 * W;
    const int patch_px0 = px_tile * PN * R - a.ph * a.W - a.pw;
    auto load_patch = [&](int base, v4i* v) {
#pragma unroll
        for (int b = 0; b < kBatch; ++b) {
            const uint32_t i = (uint32_t)min(base + b * kThreads + (int)threadIdx.x, args.patch_chunks - 1);
            const uint32_t px = fast_div(i, args.chunks_mul, args.chunks_shift), chunk = i - px * (uint32_t)(a.C16 >> 4);
            const int m = min(max(patch_px0 + (int)px, 0), (int)a.M - 1);
            v[b] = *reinterpret_cast<const v4i*>(a.x + ((uint32_t)m * (uint32_t)a.x_w_stride + chunk * 16));
        }
    };
    auto store_patch = [&](int base, const v4i* v) {
#pragma unroll
        for (int b = 0; b < kBatch; ++b) {
            const uint32_t i = (uint32_t)min(base + b * kThreads + (int)threadIdx.x, args.patch_chunks - 1);
            const uint32_t px = fast_div(i, args.chunks_mul, args.chunks_shift), chunk = i - px * (uint32_t)(a.C16 >> 4);
            v4i flipped = v[b];
#pragma unroll
            for (int e = 0; e < 4; ++e) flipped[e] ^= (int)args.x_flip;
            *reinterpret_cast<v4i*>(patch + 64 + px * (uint32_t)args.patch_pitch + chunk * 16) = flipped;
        }
    };
    v4i batch[kForm == kPatch ? kBatch : 1];
    if constexpr (kForm == kPatch) load_patch(0, batch);
    Step ring[kDepth];
    if (lo < hi) {
#pragma unroll
        for (int d = 0; d < kDepth; ++d) load_w(lo + d, ring[d]);
    }
    int32_t x_off[PN];
    uint32_t taps[PN];  // inside the image
#pragma unroll
    for (int j = 0; j < PN; ++j) {
        const int64_t m64 = (int64_t)(px_tile * PN + j) * R + col;
        const uint32_t m = (uint32_t)(m64 < a.M ? m64 : a.M - 1);  // (pixels past the end are not stored)
        if (a.px_linear) {
            x_off[j] = (int32_t)(m * (uint32_t)a.x_w_stride);
        } else {
            const uint32_t r = fast_div(m, a.ow_mul, a.ow_shift), ow = m - r * (uint32_t)a.OW;
            const uint32_t n = fast_div(r, a.oh_mul, a.oh_shift), oh = r - n * (uint32_t)a.OH;
            const int ih0 = (int)oh * a.sh - a.ph, iw0 = (int)ow * a.sw - a.pw;
            x_off[j] = (int32_t)n * (int32_t)a.x_n_stride + ih0 * (int32_t)a.x_h_stride + iw0 * (int32_t)a.x_w_stride;
            if (kForm != kPoint) {
                const int c_lo = min(max(-iw0, 0), a.KW), c_hi = min(max(a.W - iw0, 0), a.KW);
                const int r_lo = min(max(-ih0, 0), a.KH), r_hi = min(max(a.H - ih0, 0), a.KH);
                // the column bits repeated in every filter row, the rows outside the image cut off
                const uint32_t cols = c_hi > c_lo ? (uint32_t)(((uint64_t)1 << c_hi) - ((uint64_t)1 << c_lo)) : 0u;
                const uint32_t rows = r_hi > r_lo ? (uint32_t)(((uint64_t)1 << (r_hi * a.KW)) - ((uint64_t)1 << (r_lo * a.KW))) : 0u;
                taps[j] = (cols * a.row_unit) & rows;
            }
        }
        if constexpr (kForm == kPatch) x_off[j] = 64 + (j * R + col) * args.patch_pitch;
        x_off[j] += group * 16;
    }

    // the step whose pixels are loaded next: its place in its filter tap, the tap, and the offset into x
    int k_in = 0, tap = 0, kw = 0, at = lo;
    uint32_t x_at = 0;
    if constexpr (kForm != kPoint) {
        const int k = lo * kStep;
        tap = (int)fast_div((uint32_t)k, args.c64_mul, args.c64_shift);
        k_in = k - tap * a.C64;
        const int kh = (int)fast_div((uint32_t)tap, args.kw_mul, args.kw_shift);
        kw = tap - kh * a.KW;
        x_at = kForm == kPatch ? (uint32_t)((kh * a.W + kw) * args.patch_pitch + k_in) : (uint32_t)(kh * (int)a.x_h_stride + kw * (int)a.x_w_stride + k_in);
    }
    const uint32_t row_step = kForm == kPatch ? (uint32_t)((a.W - a.KW + 1) * args.patch_pitch) : (uint32_t)a.x_h_stride - (uint32_t)((a.KW - 1) * (int)a.x_w_stride);
    const uint32_t column_step = kForm == kPatch ? (uint32_t)args.patch_pitch : (uint32_t)a.x_w_stride;
    auto next_step = [&]() {
        if (at < last) {
            ++at;
            k_in += kStep;
            x_at += kStep;
            if (k_in == a.C64) {
                x_at -= (uint32_t)a.C64;
                k_in = 0;
                ++tap;
                ++kw;
                const bool row = kw == a.KW;
                kw = row ? 0 : kw;
                x_at += row ? row_step : column_step;
            }
        }
    };
    auto load_x = [&](Step& s) {
        if constexpr (kForm == kPoint) {  // (channels past C16: as below)
            const uint32_t k = (uint32_t)(at * kStep);
            at = min(at + 1, last);
#pragma unroll
            for (int j = 0; j < PN; ++j) {
                const uint32_t off = (int)k + group * 16 < a.C16 ? (uint32_t)x_off[j] + k : 0u;
                s.x[j] = *reinterpret_cast<const v4i*>(a.x + off);
            }
            return;
        }
        // channels past C16 have zero weights, and a tap outside the image becomes the zero point: both read anything inside x
        const bool channels = k_in + group * 16 < a.C16;
#pragma unroll
        for (int j = 0; j < PN; ++j) {
            const bool inside = channels && ((taps[j] >> tap) & 1);
            const uint32_t off = inside ? (uint32_t)x_off[j] + x_at : 0u;
            s.x[j] = *reinterpret_cast<const v4i*>(a.x + off);
#pragma unroll
            for (int e = 0; e < 4; ++e) s.x[j][e] = inside ? s.x[j][e] : fill;
        }
        next_step();
    };
    if constexpr (kForm != kPatch) {
        if (lo < hi) {
#pragma unroll
            for (int d = 0; d < kDepth; ++d) load_x(ring[d]);
        }
    }
    // unit u of the result: four channels of one pixel per lane (u / kQuads: block of R pixels, u % kQuads: of 8 channels);
    // this wavefront finishes units wave, wave + W, ...
    constexpr int kMine = (kUnits + W - 1) / W;
    struct Finish {
        int64_t m;
        int c0;
        int32_t add[4];    // what the zero point and an int32 bias add to the sum
        float scale[4], fbias[4];
        uint32_t r;        // residual codes
    };
    const int OC = a.oc_split > 0 && oc0 < a.oc_split ? a.oc_split : a.OC;
    auto prefetch = [&](int u, Finish& f) {
        const int j = u / kQuads, q = u % kQuads;
        f.m = (int64_t)(px_tile * PN + j) * R + col;
        f.c0 = oc0 + q * 8 + group * 4;
        const bool mine = f.m < a.M && f.c0 < OC;
        f.r = 0;
        if (a.res.r && mine) {
            const char* src = a.res.r + f.m * a.res.r_px_stride + f.c0;
            if (a.res.r_vec_ok && f.c0 + 4 <= OC) f.r = *reinterpret_cast<const uint32_t*>(src);
            else
                for (int e = 0; e < 4; ++e)
                    if (f.c0 + e < OC) f.r |= (uint32_t)(uint8_t)src[e] << (8 * e);
        }
        if (a.w_scale_len > 1 && a.OC % 4 == 0) {
            typedef int v4i_d __attribute__((ext_vector_type(4), aligned(4)));
            typedef float v4f_d __attribute__((ext_vector_type(4), aligned(4)));
            typedef const v4f_d __attribute__((address_space(1))) * Global;  // (which the compiler does not see of a choice of two)
            const int ch = min(f.c0, a.OC - 4);
            const v4i_d add = *reinterpret_cast<const v4i_d*>(a.wsum + ch);
            const v4f_d scale = *reinterpret_cast<const v4f_d*>(a.w_scale + ch), bias = *(Global)(uint64_t)((a.bias ? a.bias : a.wsum) + ch);  // (no branch around a load)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                f.add[e] = add[e];
                f.scale[e] = scale[e];
                f.fbias[e] = bias[e];
            }
            return;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int ch = min(f.c0 + e, a.OC - 1);
            f.add[e] = a.wsum[ch];
            f.scale[e] = a.w_scale_len > 1 ? a.w_scale[ch] : a.w_scale[0];
            f.fbias[e] = a.bias ? __builtin_bit_cast(float, a.bias[ch]) : 0.f;
        }
    };
    Finish mine[kMine];
#pragma unroll
    for (int i = 0; i < kMine; ++i)
        if (wave + i * W < kUnits) prefetch(wave + i * W, mine[i]);

    acc_t acc[PN];
#pragma unroll
    for (int j = 0; j < PN; ++j)
#pragma unroll
        for (int r = 0; r < 4 * kQuads; ++r) acc[j][r] = 0;
    if constexpr (kForm == kPatch) {
        if (threadIdx.x < 16) reinterpret_cast<int*>(patch)[threadIdx.x] = fill ^ (int)args.x_flip;
        store_patch(0, batch);
        for (int base = kBatch * kThreads; base < args.patch_chunks; base += kBatch * kThreads) {
            load_patch(base, batch);
            store_patch(base, batch);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    }
    auto multiply = [&](const Step& s) {
#pragma unroll
        for (int j = 0; j < PN; ++j) {
            v4i fx;
            if constexpr (kForm == kPatch) {  // (channels past C16 have zero weights: what follows a pixel's channels is some other's)
                const uint32_t off = (taps[j] >> tap) & 1 ? (uint32_t)x_off[j] + x_at : (uint32_t)(group * 16);
                fx = *reinterpret_cast<const v4i*>(patch + off);
            } else {
                fx = s.x[j];
#pragma unroll
                for (int e = 0; e < 4; ++e) fx[e] ^= (int)args.x_flip;
            }
            if constexpr (R == 32) acc[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(s.w, fx, acc[j], 0, 0, 0);
            else acc[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(s.w, fx, acc[j], 0, 0, 0);
        }
        if constexpr (kForm == kPatch) next_step();
    };
    if (lo < hi) {
        int step = lo;
        for (; step + kDepth < hi; step += kDepth) {
#pragma unroll
            for (int d = 0; d < kDepth; ++d) {
                multiply(ring[d]);
                load_w(step + d + kDepth, ring[d]);
                if constexpr (kForm != kPatch) load_x(ring[d]);
            }
        }
#pragma unroll
        for (int d = 0; d < kDepth; ++d)
            if (step + d < hi) multiply(ring[d]);
    }

    // ---- the sums, requantized ----
    const bool second = a.oc_split > 0 && oc0 >= a.oc_split;
    char* const y = second ? a.y2 - a.oc_split : a.y;
    const int64_t y_px_stride = second ? a.y2_px_stride : a.y_px_stride;
    const uint32_t y_flip = second ? a.y2_flip : a.y_flip;
    const QuantParams q_out = second ? a.q2 : a.rq.q;
    const float inv_y_scale = second ? a.inv_y_scale2 : a.inv_y_scale, lo_folded = second ? a.lo_folded2 : a.lo_folded;
    auto finish = [&](const Finish& f, v4i sum) {
        if (f.m >= a.M || f.c0 >= OC) return;
        int32_t code[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int32_t bias = __builtin_bit_cast(int32_t, f.fbias[e]);
            int32_t v = sum[e] + a.corr_mult * f.add[e];
            if (a.rq.bias_mode == kBiasOnnxInt32) v += bias;
            float x = (float)v * (a.rq.x_scale * f.scale[e]);
            if (a.rq.bias_mode == kBiasReferenceFloat) x = x + (float)bias;
            code[e] = args.rne ? quantize_value_folded<true>(x, q_out, inv_y_scale, lo_folded) : quantize_value_folded<false>(x, q_out, inv_y_scale, lo_folded);
        }
        if (a.oc_split == kFloatResults) {  // a DequantizeLinear behind the convolution
            float* dst = a.floats + f.m * a.floats_px_stride + f.c0;
            v4f out;
#pragma unroll
            for (int e = 0; e < 4; ++e) out[e] = dequantize_value(code[e], a.floats_zp, a.floats_scale);
            if (f.c0 + 4 <= OC) *reinterpret_cast<v4f_u*>(dst) = out;
            else
                for (int e = 0; e < 4; ++e)
                    if (f.c0 + e < OC) dst[e] = out[e];
            return;
        }
        uint32_t word = pack4(code[0], code[1], code[2], code[3]);
        if (a.res.r) {
            if (a.res.affine) word = affine_residual4(word, f.r, a.res);
            else word = (uint32_t)add_residual16_any(v4i{(int)word, 0, 0, 0}, v4i{(int)f.r, 0, 0, 0}, a.res)[0];
        }
        word ^= y_flip;
        char* dst = y + f.m * y_px_stride + f.c0;
        if (f.c0 + 4 <= OC) *reinterpret_cast<u32_u*>(dst) = word;
        else
            for (int e = 0; e < 4; ++e)
                if (f.c0 + e < OC) dst[e] = (char)(word >> (8 * e));
    };
    if constexpr (W > 1) {
#pragma unroll
        for (int u = 0; u < kUnits; ++u) {
            const int j = u / kQuads, q = u % kQuads;
            part[wave][u][lane] = v4i{acc[j][4 * q], acc[j][4 * q + 1], acc[j][4 * q + 2], acc[j][4 * q + 3]};
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < kMine; ++i) {
        const int u = wave + i * W;
        if (u >= kUnits) break;
        v4i sum;
        if constexpr (W > 1) {
            sum = part[0][u][lane];
#pragma unroll
            for (int w = 1; w < W; ++w) sum += part[w][u][lane];
        } else {
            const int j = i / kQuads, q = i % kQuads;
            sum = v4i{acc[j][4 * q], acc[j][4 * q + 1], acc[j][4 * q + 2], acc[j][4 * q + 3]};
        }
        finish(mine[i], sum);
    }
}

constexpr int kLdsOfUnit = 160 * 1024;

constexpr int partial_bytes(int R, int PN, int W) {
    return W > 1 ? W * PN * (R * R / 256) * 1024 : 0;
}

int patch_pitch(const ConvMfmaArgs& a) {  // an odd number of 16 bytes: neighbouring pixels on different banks (1.5 to 2 conflict cycles per LDS instruction are left)
    return a.C16 % 32 == 0 ? a.C16 + 16 : a.C16;
}

int patch_pixels(const ConvMfmaArgs& a, int tile_px) {
    return tile_px + (a.KH - 1) * a.W + a.KW - 1;
}

int patch_bytes(const ConvMfmaArgs& a, int tile_px) {
    return 64 + patch_pixels(a, tile_px) * patch_pitch(a) + 64;  // (a pixel's channels are read up to C64)
}

// kDepth: steps in flight.  All of a wavefront's steps when they are no more than eight (as far as registers allow: six of
// the largest tile, five with sixteen wavefronts): each round trip less is most of a microsecond.  ResNet-50 on one image
// 303 -> 294 us.
template <int R, int PN, int W>
int launch(const ConvMfmaArgs& a, uint32_t flip, bool rne, Form form, hipStream_t s) {
    constexpr int kDeep = R * PN == 64 ? 6 : W == 16 && PN == 2 ? 5 : 8, kStep = 1024 / R;
    const int64_t tiles = (int64_t)a.tiles_oc * a.tiles_px;
    const int per_xcd = (int)((tiles + 7) / 8);
    const int steps = (a.KP / kStep + W - 1) / W;
    ConvSplitArgs args;
    args.conv = a;
    args.x_flip = flip;
    args.rne = rne ? 1 : 0;
    args.tiles_per_xcd = per_xcd;
    magic_divisor((uint32_t)a.tiles_px, &args.tiles_px_mul, &args.tiles_px_shift);
    magic_divisor((uint32_t)a.C64, &args.c64_mul, &args.c64_shift);
    magic_divisor((uint32_t)a.KW, &args.kw_mul, &args.kw_shift);
    magic_divisor((uint32_t)(a.C16 / 16), &args.chunks_mul, &args.chunks_shift);
    args.patch_pitch = patch_pitch(a);
    args.patch_chunks = patch_pixels(a, R * PN) * (a.C16 / 16);
    const int lds = form == kPatch ? patch_bytes(a, R * PN) : 0;
#define CHX_SPLIT(FORM, DEPTH)                                                                                                                             \
    do {                                                                                                                                                   \
        if (lds + partial_bytes(R, PN, W) > 64 * 1024) /* (has to be asked for, on every device) */                                                        \
            CHX_HIP_CALL(hipFuncSetAttribute(reinterpret_cast<const void*>(&conv_split_kernel<R, PN, W, FORM, DEPTH>), hipFuncAttributeMaxDynamicSharedMemorySize, \
                                             kLdsOfUnit - partial_bytes(R, PN, W)));                                                                       \
        conv_split_kernel<R, PN, W, FORM, DEPTH><<<8 * per_xcd, 64 * W, lds, s>>>(args);                                                                   \
    } while (0)
    if (form == kPatch && steps > 5) CHX_SPLIT(kPatch, 9);  // (a step in flight is four registers: 4.5 or 9 for the layers of ResNet-50)
    else if (form == kPatch) CHX_SPLIT(kPatch, 5);
    else if (form == kTaps && steps > 4) CHX_SPLIT(kTaps, kDeep);
    else if (form == kTaps) CHX_SPLIT(kTaps, 4);
    else if (steps > 4) CHX_SPLIT(kPoint, kDeep);
    else CHX_SPLIT(kPoint, 4);
#undef CHX_SPLIT
    return launch_check("conv_split_kernel");
}

}  // namespace

bool conv_split_has(int tile_oc, int tile_px, int waves) {
    for (const ConvSplitTile& t : kConvSplitTiles)
        if (t.oc == tile_oc && t.px == tile_px && t.waves == waves) return true;
    return false;
}

// Stride 1, the results' image of the input's size, its pixels dense: a tap is a distance in pixels.  The run has to fit LDS
// beside the partial sums, and its indices 32 bits.
bool conv_split_patch_takes(const ConvMfmaArgs& a, int tile_oc, int tile_px, int waves) {
    return a.KH * a.KW > 1 && a.KH * a.KW <= 32 && a.sh == 1 && a.sw == 1 && a.OH == a.H && a.OW == a.W && a.ph < a.KH && a.pw < a.KW &&
           a.x_h_stride == (int64_t)a.W * a.x_w_stride && (a.x_n_stride == (int64_t)a.H * a.x_h_stride || a.M == (int64_t)a.OH * a.OW) &&
           a.x_w_stride >= a.C16 && (a.KH - 1) * (int64_t)a.W < 8192 && a.C16 <= 8192 &&
           (int64_t)patch_pixels(a, tile_px) * patch_pitch(a) + 128 + partial_bytes(tile_oc, tile_px / tile_oc, waves) <= kLdsOfUnit;
}

int launch_conv_split(const ConvMfmaArgs& a, int tile_oc, int tile_px, int waves, bool patch, bool x_unsigned, bool rne, hipStream_t s) {
    // a filter of one tap, inside the image for every pixel, or any filter
    const bool taps = a.KH * a.KW > 1 || a.ph != 0 || a.pw != 0 || (int64_t)(a.OH - 1) * a.sh + a.KH > a.H || (int64_t)(a.OW - 1) * a.sw + a.KW > a.W;
    const Form form = patch && conv_split_patch_takes(a, tile_oc, tile_px, waves) ? kPatch : taps ? kTaps : kPoint;
    const uint32_t flip = x_unsigned ? 0x80808080u : 0u;
#define CHX_SPLIT(R, PN, W) \
    if (tile_oc == R && tile_px == R * PN && waves == W) return launch<R, PN, W>(a, flip, rne, form, s);
    CHX_SPLIT(16, 1, 8)
    CHX_SPLIT(16, 1, 16)
    CHX_SPLIT(16, 2, 4)
    CHX_SPLIT(16, 2, 8)
    CHX_SPLIT(16, 2, 16)
    CHX_SPLIT(32, 1, 2)
    CHX_SPLIT(32, 1, 4)
    CHX_SPLIT(32, 1, 8)
    CHX_SPLIT(32, 2, 4)
    CHX_SPLIT(32, 2, 8)
#undef CHX_SPLIT
    CHX_FAIL(CHX_HIP_EINVAL, "conv_split: no kernel for a %dx%d tile with %d wavefronts", tile_oc, tile_px, waves);
}

}  // namespace chx
