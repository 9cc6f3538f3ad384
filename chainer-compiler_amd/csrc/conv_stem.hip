// Direct int8 convolution for a handful of input channels read from planar (NCHW) activations:
// the first layer of an image network (3 x 7 x 7 stride 2, 3 x 3 x 3 stride 2).
//
// With so few channels a filter tap is not a usable K slice, and expanding the activations into
// an explicit [pixels][C*KH*KW] matrix costs a pass over memory several times the size of the
// input.  Here the K axis is made of the filter *rows* instead: group g = (c, kh) contributes
// the KW consecutive input bytes of one image row, padded to KWP = 4 or 8 bytes (the weights of
// the padding bytes are zero).  A work-group copies the C x PH input rows under its 8 x 16 tile
// of output pixels into LDS once; each lane then assembles its 16 K-bytes of a
// v_mfma_i32_32x32x32_i8 operand from the LDS bytes at (row of group) * pitch + ocol * stride_w
// (aligned dword reads and a byte shift: unaligned LDS reads are slow).  The packed weights of a wavefront's 32 output
// channels sit in its registers for the whole kernel.
//
// Out-of-image bytes are filled with the activation zero point, which makes them contribute
// (zp - zp) * w = 0 (runtime/chainerx_util.cc:232-274); uint8 codes become int8 by flipping the
// top bit, and the accumulators are seeded with (128 - zp) * sum_k w[oc, k] as in conv_mfma.hip.
// The epilogue is the requantization of quant_math.h, codes transposed through a wave-private
// LDS area into [pixel][oc] rows and written as 128-bit stores to the channels-last output.
//
// The rows may be floats: then the QuantizeLinear in front of the layer happens between the load and LDS, on 1.6 times as
// many values as the image has (tiles share rows), and its pass over memory (11.6 us for 64 images of 3 x 224 x 224, 20 for
// 128) and its launch are gone.
//
// What bounds it is how long one tile takes a wavefront (some 3000 cycles by itself for 7x7 filters, of which a quarter are vector
// instructions) and the writing of the result, so everything is done to keep wavefronts independent and many: one barrier per tile, no
// wait for the next tile's rows before they go into LDS, at most 128 registers.  Measured inside a recording, with the
// QuantizeLinear: 3 -> 64 channels, 7x7, 64 images of 224 x 224 47.0 us as two launches, 38.5 as one, 8 images 11.9 and 9.7, one
// 7.7 and 7.1; 3 -> 32 channels, 3x3, 128 images 60 with the weights and constants in LDS and two barriers per tile, 50 without, 33 as
// one launch, 8 images 9.2 and 7.1.
#include <type_traits>

#include "contract.h"
#include "conv_mfma.h"

namespace chx {
namespace {

typedef int v2i __attribute__((ext_vector_type(2)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v4i_u __attribute__((ext_vector_type(4), aligned(1)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kTileH = 8;    // output rows per work-group: two per wavefront
constexpr int kTileW = 16;   // output columns
constexpr int kMaxKB = 8;    // 32-byte K blocks
constexpr int kMaxPatchDwords = 8;  // per thread: the input patch holds at most 256 * 8 dwords, counted without the columns in front (head)
constexpr int kAnyPatchDwords = 10;  // with them (as an expanded matrix and a product, and this way: 4 -> 64 channels, 3x3 filters with a stride of 4 and a padding of 1, 64
                                     // images of 224x224 35.3 and 22.1 us, 8 images 10.3 and 6.6; 3 -> 32 channels, 3x3, 64 images of 4096x3 344 and 110, one of 64x3 6.0 and 4.1)
constexpr size_t kFewPatchBytes = 256 * 3 * 4;

struct __attribute__((packed, aligned(1))) Unaligned4 {
    uint32_t v;
};
struct __attribute__((packed, aligned(4))) Floats4 {
    v4f v;
};
struct __attribute__((packed, aligned(4))) Aligned4x2 {
    v2i v;
};

// Weight repacking: w [OC][C][KH][KW] -> operand order.  Per block of 64 output channels, per
// K block kb, per 32-channel half i, lane l holds the 16 bytes  oc = i*32 + l%32,
// k = kb*32 + (l/32)*16 + 0..15  with  k = (c*KH + kh)*KWP + kw.
__global__ __launch_bounds__(256) void pack_weights_stem_kernel(
        const char* __restrict__ w, int64_t s_oc, int64_t s_c, int64_t s_kh, int64_t s_kw, int OC, int C, int KH, int KW, int KWP,
        int KB, int8_t* __restrict__ wd, int64_t total) {
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= total) return;
    const int b = (int)(idx & 15);
    const int l = (int)((idx >> 4) & 63);
    const int i = (int)((idx >> 10) & 1);
    const int64_t rest = idx >> 11;
    const int kb = (int)(rest % KB);
    const int ocblk = (int)(rest / KB);
    const int oc = ocblk * 64 + i * 32 + (l & 31);
    const int k = kb * 32 + (l >> 5) * 16 + b;
    const int g = k / KWP, kw = k % KWP;
    const int c = g / KH, kh = g % KH;
    int8_t v = 0;
    if (oc < OC && c < C && kw < KW) v = *reinterpret_cast<const int8_t*>(w + oc * s_oc + c * s_c + kh * s_kh + kw * s_kw);
    wd[idx] = v;
}

// n / d for n < 2^31 with the multiplier and shift of magic_divisor() (conv_mfma.h)
__device__ __forceinline__ uint32_t magic_div(uint32_t n, uint32_t mul, uint32_t shift) {
    return (__umulhi(n, mul) + n) >> shift;
}

// n / d for n < 2^14 and d <= 64 with m = ceil(2^20 / d)
__device__ __forceinline__ int small_div(int n, uint32_t m) {
    return (int)(((uint32_t)n * m) >> 20);
}

// Sixteen pixels of one output channel in a lane's accumulators, 32 channels in a wavefront's columns (the pixels are the first
// operand): the channel's scale and summands are one register each, and the codes go into LDS as [channel][pixel] dwords,
// from where ds_read_b64_tr_b8 brings them back as eight channels of a pixel.
__device__ __forceinline__ v2i transposed8(const char* p) {
    using Lds = __attribute__((address_space(3))) v2i*;
    return __builtin_amdgcn_ds_read_tr8_b64_v2i32((Lds)(uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)p);
}

// The reference's rounding in one of its forms and either bias, rounding to nearest even, or the one form most networks
// meet (QuantProduct::path 3, no float bias) by itself: with all forms in one kernel its scalar registers do not suffice (137 moves
// to and from lanes of vector registers, 74 this way).
enum StemRounding { kStemReference, kStemRne, kStemTwoFma };

// kKB: 32-byte K blocks held in registers, at least a.KB (the others multiply zeros: with a branch around each block its reads
// from LDS cannot run ahead of the MFMAs in front of it: 39.8 us for 35.9 at 3 -> 64 channels, 7x7, 64 images);
// kPD: patch dwords per thread (kAnyPatchDwords: also images of fewer than 4 columns); kPG: groups of 32 pixels per wavefront: 1 for up to 32 output channels, or 2, the other two
// wavefronts with the other 32 channels (one group and 64 channels each: 199 registers, two work-groups on a unit, 42 us for 39.8).
template <int KWP, int kKB, int kPD, int kPG, StemRounding kRounding, bool kFloat>
__global__ __launch_bounds__(256, 2) void conv_stem_kernel(ConvStemArgs a) {
    constexpr int GPL = 16 / KWP;  // groups per lane and K block
    constexpr int kElem = kFloat ? 4 : 1;
    using Fetched = std::conditional_t<kFloat, Floats4, Unaligned4>;
    constexpr int kStage = 1024;  // bytes per wavefront: [channel][32 pixels]
    extern __shared__ __attribute__((aligned(16))) char lds[];
    // LDS: staging [4 waves] | two patches
    char* const s_patch = lds + 4 * kStage;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = kPG == 2 ? wave & 1 : 0;  // which 32 of the block's channels
    const int oc0 = blockIdx.y * 64 + half * 32;
    const int PH = (kTileH - 1) * a.sh + a.KH;         // patch rows per channel
    const int head = -a.pw & 3;                           // the patch begins at a multiple of 4 of the image's columns, this far before the tile's
    const int PP = (head + (kTileW - 1) * a.sw + KWP + 3) & ~3;  // patch row pitch, bytes
    const int patch_dwords = a.C * PH * (PP >> 2);
    const int patch_bytes = (patch_dwords * 4 + 16 + 15) & ~15;  // the aligned reads of the last window reach one dword past it

    // the patch dwords this thread fills: the same places for every tile
    int pd_rc[kPD] = {};        // row << 16 | column
    uint32_t pd_off[kPD] = {};  // bytes from the place of the first of all channels in memory (their stride may be negative): run_conv_mfma sees to it that they fit
    const int c_turn = a.x_c_stride < 0 ? a.C - 1 : 0;
    const uint32_t c_step = (uint32_t)(a.x_c_stride < 0 ? -a.x_c_stride : a.x_c_stride);
#pragma unroll
    for (int j = 0; j < kPD; ++j) {
        const int d = tid + 256 * j;
        if (d >= patch_dwords) break;
        const int row = small_div(d, a.m_ppw), cw = d - row * (PP >> 2);
        const int c = small_div(row, a.m_ph), pr = row - c * PH;
        pd_rc[j] = pr << 16 | cw * 4;
        pd_off[j] = (uint32_t)(c_turn != 0 ? c_turn - c : c) * c_step + (uint32_t)pr * (uint32_t)a.x_h_stride + (uint32_t)(cw * 4 * kElem);
    }

    const uint32_t flip = a.x_unsigned ? 0x80808080u : 0u;
    const uint32_t fill = (uint32_t)(a.x_zp & 0xff) * 0x01010101u;
    const int tiles_per_image = a.tiles_h * a.tiles_w;
    const int npd = (patch_dwords + 255) >> 8;  // patch dwords per thread, rounded up
    // The patch of a tile is fetched into registers one tile ahead, so that the memory latency
    // runs under the previous tile's MFMAs and requantization.  A dword that reaches over the image's border is read from
    // the nearest place inside and put right on the way into LDS: nothing waits for the loads before that.
    decltype(Fetched::v) pv[kPD];
    int n = 0, oh0 = 0, ow0 = 0;  // of the tile fetched last
    int ih0 = 0, iw0 = 0;
    bool inside = false;
    const bool narrow = kPD == kAnyPatchDwords && a.W < 4;
    auto fetch_patch = [&](int t) {
        n = (int)magic_div((uint32_t)t, a.tpi_mul, a.tpi_shift);
        const int r = t - n * tiles_per_image;
        const int th = (int)magic_div((uint32_t)r, a.tw_mul, a.tw_shift), tw = r - th * a.tiles_w;
        oh0 = th * kTileH;
        ow0 = tw * kTileW;
        ih0 = oh0 * a.sh - a.ph;
        iw0 = ow0 * a.sw - a.pw - head;
        inside = ih0 >= 0 && ih0 + PH <= a.H && iw0 >= 0 && iw0 + PP <= a.W;
        const char* from = a.x + (n * a.x_n_stride + c_turn * a.x_c_stride + ih0 * a.x_h_stride + iw0 * kElem);
        // (the places past the patch are those of its first dword)
        if (inside) {
#pragma unroll
            for (int j = 0; j < kPD; ++j) {
                if (j >= npd) break;
                pv[j] = reinterpret_cast<const Fetched*>(from + pd_off[j])->v;
            }
        } else if (narrow) {  // (there are no 4 bytes to read: the row's, as the last of a dword)
            if constexpr (kPD == kAnyPatchDwords) {
#pragma unroll
                for (int j = 0; j < kPD; ++j) {
                    if (j >= npd) break;
                    const int ih = ih0 + (pd_rc[j] >> 16), iw = iw0 + (pd_rc[j] & 0xffff);
                    const char* src = from + ((int64_t)pd_off[j] + (int64_t)(min(max(ih, 0), a.H - 1) - ih) * a.x_h_stride - iw);
                    pv[j] = 0;
                    for (int e = 0; e < a.W; ++e) pv[j] |= (uint32_t)(uint8_t)src[e] << (8 * (4 - a.W + e));
                }
            }
        } else {
#pragma unroll
            for (int j = 0; j < kPD; ++j) {
                if (j >= npd) break;
                const int ih = ih0 + (pd_rc[j] >> 16), iw = iw0 + (pd_rc[j] & 0xffff);
                const int64_t move = (int64_t)(min(max(ih, 0), a.H - 1) - ih) * a.x_h_stride + (min(max(iw, 0), a.W - 4) - iw) * kElem;
                const char* src = from + ((int64_t)pd_off[j] + move);
                pv[j] = reinterpret_cast<const Fetched*>(src)->v;
            }
        }
    };
    QuantProduct xq;
    if (kFloat) xq = in_vector_registers(a.xq);
    auto put_patch = [&](char* patch) {
#pragma unroll
        for (int j = 0; j < kPD; ++j) {
            if (j >= npd) break;
            uint32_t v;
            if constexpr (kFloat) {
                // (below 256 also where it is not a number, as the comparison with the largest code has it; the two parts of
                // the reciprocal have one sign, so that infinities stay what they are)
                float t[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) t[e] = __builtin_fminf(quantize_prefloor_u8<1>(pv[j][e], xq), 256.f);
                v = floor_sat_u8x4(t[0], t[1], t[2], t[3]);
            } else {
                v = pv[j];
            }
            if (!inside) {
                const int ih = ih0 + (pd_rc[j] >> 16), iw = iw0 + (pd_rc[j] & 0xffff);
                const int n_in = (unsigned)ih < (unsigned)a.H && iw >= 0 ? min(max(a.W - iw, 0), 4) : 0;  // bytes inside: the last of those read
                if (n_in < 4) v = n_in == 0 ? fill : (v >> (32 - 8 * n_in)) | fill << (8 * n_in);
            }
            if (tid + 256 * j < patch_dwords) reinterpret_cast<uint32_t*>(patch)[tid + 256 * j] = v ^ flip;
        }
    };
    // The device deals work-groups out to its 8 XCDs in turn: the work-groups of XCD x (blockIdx.x % 8 == x; the grid's
    // x extent is a multiple of 8) share the tiles [x * chunk, (x + 1) * chunk), so that the input rows neighbouring tiles
    // have in common (15 of a tile's 21 rows for a 7x7 filter with stride 2) are found in that XCD's own L2.
    const int t_step = (int)(gridDim.x >> 3);
    const int chunk = (a.tiles + 7) >> 3;
    const int t_first = (int)(blockIdx.x & 7u) * chunk + (int)(blockIdx.x >> 3);
    const int t_end = min(((int)(blockIdx.x & 7u) + 1) * chunk, a.tiles);
    if (t_first >= t_end) return;
    fetch_patch(t_first);

    // the weights of this block of output channels, already in operand order
    v4i fw[kKB];
    {
        const v4i* src = reinterpret_cast<const v4i*>(a.wd + (int64_t)blockIdx.y * a.KB * 2048);
#pragma unroll
        for (int kb = 0; kb < kKB; ++kb)
            fw[kb] = kb < a.KB ? src[(kb * 2 + half) * 64 + lane] : v4i{0, 0, 0, 0};
    }
    // what belongs to the lane's output channel (the loads first: nothing waits between them)
    const int my_oc = min(oc0 + (lane & 31), a.OC - 1);
    const int32_t wsum = a.wsum[my_oc], bias = a.bias ? a.bias[my_oc] : 0;
    const float w_scale = a.w_scale[a.w_scale_len > 1 ? my_oc : 0];

    // LDS offsets of this lane's K groups, relative to the patch: group row + pixel position
    const int p = lane & 31;
    const int group0 = kPG == 2 ? wave & 2 : wave;  // the wavefront's first group: two rows of the tile
    const int orow = 2 * group0 + (p >> 4), ocol = p & 15;
    const int kq = lane >> 5;
    int offs[kKB][GPL];
    {
        const int G = a.C * a.KH;
        const int loff = orow * a.sh * PP + head + ocol * a.sw;
#pragma unroll
        for (int kb = 0; kb < kKB; ++kb)
#pragma unroll
            for (int j = 0; j < GPL; ++j) {
                int g = kb * (32 / KWP) + kq * GPL + j;
                g = g < G ? g : G - 1;  // padding groups have zero weights; read something valid
                const int c = small_div(g, a.m_kh), kh = g - c * a.KH;
                offs[kb][j] = ((c * PH + kh) * PP + loff) & ~3;
            }
    }
    const uint32_t phase = (uint32_t)(head + ocol * a.sw) & 3u;  // the pitch and the group rows are multiples of 4
    // Staging: dword kq of granule g (8 pixels) of a channel's row lies in granule g ^ (channel / 8): neither side has bank
    // conflicts.  Back come 16 pixels and twice 8 channels for each group of 16 lanes.
    char* const my_stage = lds + wave * kStage;
    const int put = (lane & 31) * 32 + kq * 4, put_x = (lane >> 3) & 3;
    const int got_chunk = (lane >> 4) & 1;  // 16 channels
    const int got_row = lane >> 5;          // of the group's two
    const int got = (got_chunk * 16 + ((lane & 15) >> 1)) * 32 + (((2 * got_row + (lane & 1)) ^ (2 * got_chunk)) << 3);

    const float scale = a.rq.x_scale * w_scale;
    const float fbias = a.rq.bias_mode == kBiasReferenceFloat ? (float)bias : 0.f;
    const int32_t add = a.corr_mult * wsum + (a.rq.bias_mode == kBiasOnnxInt32 ? bias : 0);
    // the lane's place in a group's two rows of results
    const int64_t y_row = (int64_t)a.OW * a.y_px_stride, y_lane = got_row * y_row + (lane & 15) * a.y_px_stride + got_chunk * 16;
    const int oc = oc0 + got_chunk * 16;
    put_patch(s_patch);
    __syncthreads();
    int buffer = 0;
    // (one barrier per tile: the next tile's patch goes into the other buffer, which was last read before the previous barrier)
    for (int t = t_first; t < t_end; t += t_step) {
        const int oh_t = oh0, ow_t = ow0;
        char* const y_tile = a.y + ((((int64_t)n * a.OH + oh0) * a.OW + ow0) * a.y_px_stride + oc0);
        const bool more = t + t_step < t_end;
        if (more) fetch_patch(t + t_step);
#pragma unroll
        for (int pg = 0; pg < kPG; ++pg) {
            const char* const from = s_patch + buffer * patch_bytes + pg * 2 * a.sh * PP;
            // lane holds, per 32x32 MFMA tile: output channel lane % 32, pixel rows (v/4)*8 + (lane>>5)*4 + v%4
            v16i acc;
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[e] = add;
#pragma unroll
            for (int kb = 0; kb < kKB; ++kb) {
                // the lane's window starts at any byte: read the aligned dwords around it and shift
                v4i fb;
                if (KWP == 8) {
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        const char* src = from + offs[kb][j];
                        const v2i d01 = reinterpret_cast<const Aligned4x2*>(src)->v;
                        const int d2 = *reinterpret_cast<const int*>(src + 8);
                        fb[2 * j] = (int)__builtin_amdgcn_alignbyte((uint32_t)d01[1], (uint32_t)d01[0], phase);
                        fb[2 * j + 1] = (int)__builtin_amdgcn_alignbyte((uint32_t)d2, (uint32_t)d01[1], phase);
                    }
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const v2i d01 = reinterpret_cast<const Aligned4x2*>(from + offs[kb][j % GPL])->v;
                        fb[j] = (int)__builtin_amdgcn_alignbyte((uint32_t)d01[1], (uint32_t)d01[0], phase);
                    }
                }
                acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(fb, fw[kb], acc, 0, 0, 0);
            }

            // requantize into the wave's staging rows
            // (kPath: QuantProduct::path)
            auto requantize_tile = [&](auto float_bias_tag, auto path_tag) {
                constexpr bool kFloatBias = decltype(float_bias_tag)::value;
                constexpr int kPath = decltype(path_tag)::value;
                QuantProduct qp;
                if (kPath != 0) qp = in_vector_registers(a.qp);
                uint32_t codes[4];
                float pre[16];
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    int32_t code[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        float v = (float)acc[g * 4 + e] * scale;
                        if (kFloatBias) v = v + fbias;
                        if (kPath == 0) code[e] = quantize_value_folded<kRounding == kStemRne>(v, a.rq.q, a.inv_y_scale, a.lo_folded);
                        else pre[g * 4 + e] = quantize_prefloor_u8<kPath>(v, qp);
                    }
                    if (kPath == 0) codes[g] = pack4(code[0], code[1], code[2], code[3]);
                }
                if (kPath != 0) floor_sat_u8x16(pre, codes);
#pragma unroll
                for (int g = 0; g < 4; ++g) *reinterpret_cast<uint32_t*>(my_stage + put + ((g ^ put_x) << 3)) = codes[g];
            };
            {
                using P0 = std::integral_constant<int, 0>;
                using P1 = std::integral_constant<int, 1>;
                using P2 = std::integral_constant<int, 2>;
                using P3 = std::integral_constant<int, 3>;
                const bool float_bias = a.rq.bias_mode == kBiasReferenceFloat;
                if (kRounding == kStemTwoFma) {
                    requantize_tile(std::false_type(), P3());
                } else if (kRounding == kStemRne || a.qp.path == 0) {
                    if (float_bias) requantize_tile(std::true_type(), P0());
                    else requantize_tile(std::false_type(), P0());
                } else if (a.qp.path == 2) {
                    if (float_bias) requantize_tile(std::true_type(), P2());
                    else requantize_tile(std::false_type(), P2());
                } else if (a.qp.path == 3) {
                    if (float_bias) requantize_tile(std::true_type(), P3());
                    else requantize_tile(std::false_type(), P3());
                } else {
                    if (float_bias) requantize_tile(std::true_type(), P1());
                    else requantize_tile(std::false_type(), P1());
                }
            }
            // (in front of the stores: the wait for the fetched dwords would otherwise wait for them too)
            if (pg == kPG - 1 && more) put_patch(s_patch + (buffer ^ 1) * patch_bytes);
            // the staging rows are private to the wave: its own LDS operations complete in order
            const v2i lo = transposed8(my_stage + got), hi = transposed8(my_stage + (got ^ 8) + 256);
            if (oh_t + 2 * (group0 + pg) + got_row < a.OH && ow_t + (lane & 15) < a.OW && oc < a.OC) {
                char* dst = y_tile + 2 * (group0 + pg) * y_row + y_lane;
                const v4i val = {lo[0], lo[1], hi[0], hi[1]};
                if (oc + 16 <= a.OC) {
                    *reinterpret_cast<v4i_u*>(dst) = val;
                } else {
#pragma unroll
                    for (int e = 0; e < 16; ++e)
                        if (oc + e < a.OC) dst[e] = (char)((uint32_t)val[e >> 2] >> (8 * (e & 3)));
                }
            }
        }
        if (more) __syncthreads();
        buffer ^= 1;
    }
}

}  // namespace

int stem_k_blocks(int C, int KH, int KW) {
    const int kwp = KW <= 4 ? 4 : 8;
    return (C * KH * kwp + 31) / 32;
}

int stem_patch_rows(int KH, int sh) {
    return (kTileH - 1) * sh + KH;
}

size_t stem_patch_bytes(int C, int KH, int KW, int sh, int sw, int pw) {
    const int kwp = KW <= 4 ? 4 : 8;
    const int PP = ((-pw & 3) + (kTileW - 1) * sw + kwp + 3) & ~3;
    return (size_t)C * stem_patch_rows(KH, sh) * PP;
}

bool stem_shape_fits(int C, int KH, int KW) {
    return KW <= 8 && C * KH <= 32 && stem_k_blocks(C, KH, KW) <= kMaxKB;
}

bool stem_patch_is_small(int C, int KH, int KW, int sh, int sw, int pw) {
    return stem_patch_bytes(C, KH, KW, sh, sw, pw) <= kFewPatchBytes;
}

bool stem_patch_fits(int C, int KH, int KW, int sh, int sw) {
    const int kwp = KW <= 4 ? 4 : 8;
    // the small_div ranges: rows per channel below 64, dwords per row at most 64
    return stem_patch_bytes(C, KH, KW, sh, sw, 0) <= (size_t)256 * kMaxPatchDwords * 4 && stem_patch_rows(KH, sh) < 64 && (kTileW - 1) * sw + kwp < 252;
}

int pack_weights_stem(const chx_hip_tensor& w, int OCpad64, int8_t* wd, hipStream_t s) {
    const int C = (int)w.shape[1], KH = (int)w.shape[2], KW = (int)w.shape[3];
    const int KB = stem_k_blocks(C, KH, KW);
    const int64_t total = (int64_t)(OCpad64 / 64) * KB * 2048;
    pack_weights_stem_kernel<<<(unsigned)((total + 255) / 256), 256, 0, s>>>(
            static_cast<const char*>(w.data), w.strides[0], w.strides[1], w.strides[2], w.strides[3], (int)w.shape[0], C, KH, KW,
            KW <= 4 ? 4 : 8, KB, wd, total);
    return launch_check("pack_weights_stem_kernel");
}

template <int KWP, int kKB, int kPD, int kPG, StemRounding kRounding, bool kFloat>
static int launch_stem(const ConvStemArgs& a, size_t patch, hipStream_t s) {
    // (the aligned reads of the last window reach one dword past the patch)
    const size_t lds = (size_t)4 * 1024 + 2 * ((patch + 16 + 15) / 16 * 16);
    static int cus = 0;
    if (cus == 0) {
        int dev = 0;
        hipDeviceProp_t prop;
        cus = 256;
        if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess) cus = prop.multiProcessorCount;
    }
    // as many work-groups as the device holds at once, each walking over tiles with the weights resident
    int per_cu = 0;
    const void* fn = reinterpret_cast<const void*>(&conv_stem_kernel<KWP, kKB, kPD, kPG, kRounding, kFloat>);
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, 256, lds) != hipSuccess || per_cu < 1) per_cu = 2;
    const int oc_blocks = (a.OC + 63) / 64;
    int per_block = cus * per_cu / oc_blocks;
    if (per_block < 1) per_block = 1;
    // (a multiple of 8 work-groups along x: see the kernel's tile order; and no more than it takes for the same number of
    // tiles each: with 7 for some and 6 for the others the others only slow the first down)
    const int chunk = (a.tiles + 7) / 8, at_most = (per_block + 7) / 8, rounds = chunk > at_most ? (chunk + at_most - 1) / at_most : 1;
    const int along_x = (chunk + rounds - 1) / rounds * 8;
    const dim3 grid((unsigned)along_x, (unsigned)oc_blocks);
    conv_stem_kernel<KWP, kKB, kPD, kPG, kRounding, kFloat><<<grid, 256, lds, s>>>(a);
    return launch_check("conv_stem_kernel");
}

int launch_conv_stem(ConvStemArgs a, bool rne, hipStream_t s) {
    a.tiles_h = (a.OH + kTileH - 1) / kTileH;
    a.tiles_w = (a.OW + kTileW - 1) / kTileW;
    const int64_t tiles = (int64_t)a.N * a.tiles_h * a.tiles_w;
    CHX_REQUIRE(tiles < (int64_t(1) << 30), "QLinearConv: too many output tiles for the planar-input kernel");
    a.tiles = (int32_t)tiles;
    magic_divisor((uint32_t)(a.tiles_h * a.tiles_w), &a.tpi_mul, &a.tpi_shift);
    magic_divisor((uint32_t)a.tiles_w, &a.tw_mul, &a.tw_shift);
    a.KB = stem_k_blocks(a.C, a.KH, a.KW);
    const bool kwp4 = a.KW <= 4;
    const uint32_t ppw = (uint32_t)((((-a.pw & 3) + (kTileW - 1) * a.sw + (kwp4 ? 4 : 8) + 3) & ~3) >> 2), ph_rows = (uint32_t)stem_patch_rows(a.KH, a.sh);
    a.m_ppw = ((1u << 20) + ppw - 1) / ppw;
    a.m_ph = ((1u << 20) + ph_rows - 1) / ph_rows;
    a.m_kh = ((1u << 20) + (uint32_t)a.KH - 1) / (uint32_t)a.KH;
    const size_t patch = stem_patch_bytes(a.C, a.KH, a.KW, a.sh, a.sw, a.pw);
    const bool two = a.OC > 32;
    const StemRounding rounding = rne ? kStemRne : a.qp.path == 3 && a.rq.bias_mode != kBiasReferenceFloat ? kStemTwoFma : kStemReference;
#define CHX_STEM_OF(KWP, KB, PD, ROUNDING, FLOAT) \
    (two ? launch_stem<KWP, KB, PD, 2, ROUNDING, FLOAT>(a, patch, s) : launch_stem<KWP, KB, PD, 1, ROUNDING, FLOAT>(a, patch, s))
#define CHX_STEM(KWP, KB, PD, FLOAT) \
    (rounding == kStemTwoFma && PD == 3 ? CHX_STEM_OF(KWP, KB, 3, kStemTwoFma, FLOAT) : CHX_STEM_OF(KWP, KB, PD, kStemReference, FLOAT))
    CHX_REQUIRE(!a.x_float || (patch <= kFewPatchBytes && a.W >= 4), "QLinearConv: the input rows of a tile are too many, or too short, to be quantized on the way");
    if (patch > (size_t)256 * kMaxPatchDwords * 4 || a.W < 4) {
        if (rne) return kwp4 ? CHX_STEM_OF(4, 4, kAnyPatchDwords, kStemRne, false) : CHX_STEM_OF(8, 8, kAnyPatchDwords, kStemRne, false);
        return kwp4 ? CHX_STEM(4, 4, kAnyPatchDwords, false) : CHX_STEM(8, 8, kAnyPatchDwords, false);
    }
    if (patch > kFewPatchBytes) {
        if (rne) return kwp4 ? CHX_STEM_OF(4, 4, 8, kStemRne, false) : CHX_STEM_OF(8, 8, 8, kStemRne, false);
        return kwp4 ? CHX_STEM(4, 4, 8, false) : CHX_STEM(8, 8, 8, false);
    }
    if (a.x_float) {
        if (kwp4) return a.KB <= 2 ? CHX_STEM(4, 2, 3, true) : CHX_STEM(4, 4, 3, true);
        return a.KB <= 6 ? CHX_STEM(8, 6, 3, true) : CHX_STEM(8, 8, 3, true);
    }
    if (rne) return kwp4 ? CHX_STEM_OF(4, 4, 3, kStemRne, false) : CHX_STEM_OF(8, 8, 3, kStemRne, false);
    if (kwp4) return a.KB <= 2 ? CHX_STEM(4, 2, 3, false) : CHX_STEM(4, 4, 3, false);
    return a.KB <= 6 ? CHX_STEM(8, 6, 3, false) : CHX_STEM(8, 8, 3, false);
#undef CHX_STEM
#undef CHX_STEM_OF
}

}  // namespace chx
