// The packed-weight convolution for 1x1 filters over few channels (at most 256): pixels stream past weights kept in LDS.
//
// Such a layer moves more bytes than it multiplies: 16 -> 96 channels over 128 images of 112 x 112 read 26 MB and write
// 154 MB for 2.5 G products.  conv_mfma_kernel stages the pixels in LDS, transposes the codes through LDS and meets at
// two barriers per tile of one or two K steps; what it waits for there is most of its time.  Here the work-group puts its
// weights into LDS once, in the order in which the lanes of an MFMA read them, and then each wavefront goes its own way:
// 32 pixels at a time, their K bytes straight into registers (requested one block ahead), 64 channels of codes per step,
// transposed between the lanes by four register swaps and stored as 64 contiguous bytes of each of 16 pixels.
// That example: 61 us with the staged tiles, 42 here (180 MB); 32 -> 16 channels of the same images 32 and 18 (77 MB); 144 ->
// 24 with a residual sum over 56 x 56 33 and 21.  With many channels out, the vector instructions of the requantization
// bound it (seven to nine per code), else memory.
//
// Arguments, requantization, residual sums, pairs and storage are those of conv_mfma_kernel.
#include <type_traits>

#include "conv_mfma.h"
#include "conv_device.h"

namespace chx {
namespace {

constexpr int kWaves = 4, kPixels = 32;   // per work-group; per wavefront and step: two MFMA columns of 16
constexpr int kWeightBytes = 32768;       // of a work-group's channels: four work-groups share a compute unit's 160 KB

// word t of lane group g (four channels of the pixel, channels t*16 + g*4 ..) -> the sixteen channels of tile g
__device__ __forceinline__ v4i transpose_groups(uint32_t w0, uint32_t w1, uint32_t w2, uint32_t w3) {
    const auto a = __builtin_amdgcn_permlane32_swap(w0, w2, false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(w1, w3, false, false);
    const auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
    const auto d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
    return v4i{(int)c[0], (int)c[1], (int)d[0], (int)d[1]};
}

// The first n (1 to 15) of sixteen bytes, at any alignment.
__device__ __forceinline__ void store_part(char* dst, v4i v, int n) {
    uint32_t w[4] = {(uint32_t)v[0], (uint32_t)v[1], (uint32_t)v[2], (uint32_t)v[3]};
    if (n & 8) {
        __builtin_memcpy(dst, w, 8);
        dst += 8;
        w[0] = w[2];
        w[1] = w[3];
    }
    if (n & 4) {
        __builtin_memcpy(dst, w, 4);
        dst += 4;
        w[0] = w[1];
    }
    for (int e = 0; e < (n & 3); ++e) dst[e] = (char)(w[0] >> (8 * e));
}

__device__ __forceinline__ v4i load_part(const char* src, int n) {
    uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
    for (int e = 0; e < 16; ++e)
        if (e < n) w[e / 4] |= (uint32_t)(uint8_t)src[e] << (8 * (e % 4));
    return v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
}

struct ConvPointArgs {
    ConvMfmaArgs conv;
    uint32_t x_flip;
    int32_t rne, chunks, chunk_tiles, slots;  // slots: work-groups per chunk
    uint32_t chunks_mul, chunks_shift;        // magic_divisor(chunks)
};

// kPath: QuantProduct::path (2 also for a pair of which one is 1; both are 3 or none)
template <int KS, int kPath, bool kFloatBias, bool kRes>
__global__ __launch_bounds__(64 * kWaves, 2) void conv_point_kernel(ConvPointArgs) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const ConvPointArgs& args = kernel_arguments<ConvPointArgs>();
    const ConvMfmaArgs& a = args.conv;
    const int rne = args.rne, chunks = args.chunks, chunk_tiles = args.chunk_tiles, slots = args.slots;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, group = lane >> 4;
    // the chunks of channels over one run of pixels are neighbours on one XCD: its L2 hands them the pixels
    const int turn = (int)(blockIdx.x >> 3), round = (int)fast_div((uint32_t)turn, args.chunks_mul, args.chunks_shift);
    const int chunk = turn - round * chunks, slot = round * 8 + (int)(blockIdx.x & 7);
    const int tile0 = chunk * chunk_tiles, tiles = min(chunk_tiles, (a.OC + 15) / 16 - tile0);

    // ---- this chunk's weights and constants ----
    v4i* s_w = reinterpret_cast<v4i*>(lds);  // [tile][K step][lane]
    int32_t* s_add = reinterpret_cast<int32_t*>(lds + chunk_tiles * KS * 1024);
    float* s_scale = reinterpret_cast<float*>(s_add + chunk_tiles * 16);
    float* s_fbias = s_scale + chunk_tiles * 16;
    const int bk_shift = a.bk == 128 ? 7 : 6;
    for (int i = tid; i < tiles * KS * 64; i += 64 * kWaves) {
        const int l = i & 63, ts = i >> 6, oc = (tile0 + ts / KS) * 16 + (l & 15), k = (ts % KS) * 64 + (l >> 4) * 16;
        s_w[i] = *reinterpret_cast<const v4i*>(a.wp + (int64_t)(oc >> 6) * 64 * a.KP + ((k >> bk_shift) * 64 << bk_shift) + ((oc & 63) << bk_shift) + (k & (a.bk - 1)));
    }
    for (int i = tid; i < tiles * 16; i += 64 * kWaves) {
        const int ch = min(tile0 * 16 + i, a.OC - 1);
        const int32_t bias = a.bias ? a.bias[ch] : 0;
        s_add[i] = a.corr_mult * a.wsum[ch] + (a.rq.bias_mode == kBiasOnnxInt32 ? bias : 0);
        s_scale[i] = a.rq.x_scale * (a.w_scale_len > 1 ? a.w_scale[ch] : a.w_scale[0]);
        s_fbias[i] = (float)bias;
    }
    __syncthreads();

    // ---- pixels ----
    const int blocks = (int)((a.M + kPixels - 1) / kPixels), step = slots * kWaves;
    const uint32_t pitch = (uint32_t)a.x_w_stride;
    uint32_t in_px[KS];  // channels past C16 have zero weights: any byte of the pixel stands for them
#pragma unroll
    for (int k = 0; k < KS; ++k) in_px[k] = k * 64 + group * 16 < a.C16 ? (uint32_t)(k * 64 + group * 16) : 0u;
    v4i next[2][KS];
    auto load = [&](int block) {
        const uint32_t m0 = (uint32_t)min(block, blocks - 1) * kPixels;
        const char* base = a.x + (uint64_t)m0 * pitch;
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const uint32_t px = min((uint32_t)(p * 16 + col), (uint32_t)(a.M - 1) - m0);
#pragma unroll
            for (int k = 0; k < KS; ++k) next[p][k] = *reinterpret_cast<const v4i*>(base + (px * pitch + in_px[k]));
        }
    };
    int block = slot * kWaves + wave;
    load(block);
    const int flip = (int)in_vector_register(args.x_flip);
    for (; block < blocks; block += step) {
        v4i x[2][KS];
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int k = 0; k < KS; ++k) x[p][k] = next[p][k] ^ flip;
        load(block + step);
        const int64_t m0 = (int64_t)block * kPixels;
        auto channels64 = [&](int t0, auto full_tag) {
            constexpr bool kFull = decltype(full_tag)::value;  // all four tiles are there
            const int oc0 = (tile0 + t0) * 16;
            char* y = a.y;
            int64_t y_pitch = a.y_px_stride;
            QuantParams q = a.rq.q;
            float inv = a.inv_y_scale, lo = a.lo_folded;
            QuantProduct qp = a.qp;
            uint32_t y_flip = a.y_flip;
            int OC = a.OC;
            if (a.oc_split > 0) {
                if (oc0 >= a.oc_split) {
                    y = a.y2 - a.oc_split;
                    y_pitch = a.y2_px_stride;
                    q = a.q2;
                    inv = a.inv_y_scale2;
                    lo = a.lo_folded2;
                    qp = a.qp2;
                    y_flip = a.y2_flip;
                } else {
                    OC = a.oc_split;
                }
            }
            const int ch = oc0 + group * 16, valid = OC - ch;
            v4i res[2];
            if constexpr (kRes) {
#pragma unroll
                for (int p = 0; p < 2; ++p) {
                    const int64_t m = m0 + p * 16 + col;
                    const char* src = a.res.r + m * a.res.r_px_stride + ch;
                    res[p] = v4i{0, 0, 0, 0};
                    // (an aligned chunk that holds one byte of the tensor can be read whole)
                    if (m < a.M && (valid >= 16 || (valid > 0 && a.res.r_vec_ok))) __builtin_memcpy(&res[p], src, 16);
                    else if (m < a.M && valid > 0) res[p] = load_part(src, valid);
                }
            }
            if (kPath == 0) {
                q = in_vector_registers(q);
                inv = in_vector_register(inv);
                lo = in_vector_register(lo);
            } else {
                qp = in_vector_registers(qp);
            }
            uint32_t word[2][4];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                word[0][t] = word[1][t] = 0;
                if (!kFull && t0 + t >= tiles) continue;
                const int i0 = (t0 + t) * 16 + group * 4;
                const v4i add = *reinterpret_cast<const v4i*>(&s_add[i0]);
                v4i acc[2] = {add, add};
#pragma unroll
                for (int k = 0; k < KS; ++k) {
                    const v4i w = s_w[((t0 + t) * KS + k) * 64 + lane];
#pragma unroll
                    for (int p = 0; p < 2; ++p) acc[p] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w, x[p][k], acc[p], 0, 0, 0);
                }
                const v4f sc = *reinterpret_cast<const v4f*>(&s_scale[i0]);
                v4f fb = {0.f, 0.f, 0.f, 0.f};
                if (kFloatBias) fb = *reinterpret_cast<const v4f*>(&s_fbias[i0]);
                float pre[8];
                int32_t code[8];
#pragma unroll
                for (int p = 0; p < 2; ++p)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        float v = (float)acc[p][e] * sc[e];
                        if (kFloatBias) v = v + fb[e];
                        if (kPath == 0) code[p * 4 + e] = rne ? quantize_value_folded<true>(v, q, inv, lo) : quantize_value_folded<false>(v, q, inv, lo);
                        else pre[p * 4 + e] = quantize_prefloor_u8<kPath>(v, qp);
                    }
                if (kPath == 0) {
                    word[0][t] = pack4(code[0], code[1], code[2], code[3]);
                    word[1][t] = pack4(code[4], code[5], code[6], code[7]);
                } else {
                    floor_sat_u8x8(pre, &word[0][t], &word[1][t]);
                }
            }
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                v4i val = transpose_groups(word[p][0], word[p][1], word[p][2], word[p][3]);
                if constexpr (kRes) {
                    if (a.res.affine == 1) val = affine_residual16<false>(val, res[p], a.res);
                    else if (a.res.affine == 2) val = affine_residual16<true>(val, res[p], a.res);
                    else val = add_residual16_any(val, res[p], a.res);
                }
                val ^= (int)y_flip;
                const int64_t m = m0 + p * 16 + col;
                char* dst = y + m * y_pitch + ch;
                if (m >= a.M) continue;
                if (valid >= 16) __builtin_memcpy(dst, &val, 16);
                else if (valid > 0) store_part(dst, val, valid);
            }
        };
        int t0 = 0;
        for (; t0 + 4 <= tiles; t0 += 4) channels64(t0, std::true_type());
        if (t0 < tiles) channels64(t0, std::false_type());
    }
}

template <int KS, int kPath, bool kFloatBias, bool kRes>
int launch(const ConvMfmaArgs& a, int max_wgs_per_cu, uint32_t flip, bool rne, hipStream_t s) {
    const int groups = (a.OC + 63) / 64, fit = kWeightBytes / (KS * 64 * 64);
    const int chunks = (groups + fit - 1) / fit, chunk_tiles = ((groups + chunks - 1) / chunks) * 4;
    const size_t bytes = (size_t)chunk_tiles * (KS * 1024 + 16 * 12);
    const int per_cu = max_wgs_per_cu > 0 ? max_wgs_per_cu : 4;
    // pixel slots: no more than there are blocks for, a multiple of the 8 XCDs
    const int64_t wanted = ((a.M + kPixels - 1) / kPixels + kWaves - 1) / kWaves;
    int64_t slots = 256 * per_cu / chunks;
    if (slots > wanted) slots = wanted;
    slots = (slots + 7) / 8 * 8;
    ConvPointArgs args;
    args.conv = a;
    args.x_flip = flip;
    args.rne = rne ? 1 : 0;
    args.chunks = chunks;
    args.chunk_tiles = chunk_tiles;
    args.slots = (int)slots;
    magic_divisor((uint32_t)chunks, &args.chunks_mul, &args.chunks_shift);
    conv_point_kernel<KS, kPath, kFloatBias, kRes><<<(int)(slots * chunks), 64 * kWaves, bytes, s>>>(args);
    return launch_check("conv_point_kernel");
}

template <int KS>
int launch_steps(const ConvMfmaArgs& a, int max_wgs_per_cu, uint32_t flip, bool rne, hipStream_t s) {
    const bool product = a.qp.path != 0 && (a.oc_split == 0 || a.qp2.path != 0);
    const bool two_fma = a.qp.path == 3;  // (of a pair, both)
    const bool bound = a.qp.path == 2 || (a.oc_split > 0 && a.qp2.path == 2);
    const bool fb = a.rq.bias_mode == kBiasReferenceFloat, res = a.res.r != nullptr;
#define CHX_POINT(PATH, FB) \
    return res ? launch<KS, PATH, FB, true>(a, max_wgs_per_cu, flip, rne, s) : launch<KS, PATH, FB, false>(a, max_wgs_per_cu, flip, rne, s)
    if (!product) CHX_POINT(0, true);
    if (two_fma && fb) CHX_POINT(3, true);
    if (two_fma) CHX_POINT(3, false);
    if (bound && fb) CHX_POINT(2, true);
    if (bound) CHX_POINT(2, false);
    if (fb) CHX_POINT(1, true);
    CHX_POINT(1, false);
#undef CHX_POINT
}

}  // namespace

int launch_conv_point(const ConvMfmaArgs& a, int max_wgs_per_cu, bool x_unsigned, bool rne, hipStream_t s) {
    const uint32_t flip = x_unsigned ? 0x80808080u : 0u;
    switch (a.KP / 64) {
        case 1: return launch_steps<1>(a, max_wgs_per_cu, flip, rne, s);
        case 2: return launch_steps<2>(a, max_wgs_per_cu, flip, rne, s);
        case 3: return launch_steps<3>(a, max_wgs_per_cu, flip, rne, s);
        case 4: return launch_steps<4>(a, max_wgs_per_cu, flip, rne, s);
    }
    CHX_FAIL(CHX_HIP_EINVAL, "conv_point: no kernel for %d bytes of K", a.KP);
}

}  // namespace chx
