// Depthwise 3x3 QLinearConv on NCHW arrays (rows contiguous), with the packed weights of depthwise.hip.
//
// A thread computes four neighbouring pixels of kRows output rows of one channel.  Per input row it reads the bytes under
// them in one or two 8-byte accesses at whatever alignment (columns outside the image filled in), shifts out the three
// bytes of each pixel and multiplies them with the filter row in one v_dot4_i32_i8: no layout change, no LDS, neighbouring
// lanes on neighbouring bytes.  Arithmetic and requantization are those of depthwise.hip.
// [16, 144, 56, 56]: 231 us with one thread per result (conv_direct_kernel), 7.9 here.
#include "contract.h"
#include "depthwise.h"
#include "conv_mfma.h"
#include "conv_device.h"
#include "gemm_i8_device.h"

namespace chx {
namespace {

constexpr int kRows = 4;

// columns at .. at+7 of a row shorter than 8
__device__ __forceinline__ uint64_t narrow_window(const char* row, int at, int W, uint64_t zp) {
    uint64_t v = zp;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int w = at + e;
        if (w < 0 || w >= W) continue;
        v = (v & ~((uint64_t)0xff << (8 * e))) | (uint64_t)(uint8_t)row[w] << (8 * e);
    }
    return v;
}

struct DepthwisePlanarArgs {
    DepthwiseArgs conv;
    int32_t rne, G, RB, channels;
    uint32_t g_mul, g_shift, rb_mul, rb_shift, c_mul, c_shift;
};

// S: stride.  kPath: QuantProduct::path.
template <int S, int kPath, bool kFloatBias>
__global__ __launch_bounds__(256) void depthwise_planar_kernel(DepthwisePlanarArgs) {
    const DepthwisePlanarArgs args = kernel_arguments<DepthwisePlanarArgs>();
    const DepthwiseArgs& a = args.conv;
    const int rne = args.rne;
    // (image, channel, run of rows, group of four columns), the last one fastest
    const uint32_t idx = blockIdx.x * 256u + threadIdx.x;
    const uint32_t t = fast_div(idx, args.g_mul, args.g_shift), gc = idx - t * (uint32_t)args.G;
    const uint32_t nc = fast_div(t, args.rb_mul, args.rb_shift), rb = t - nc * (uint32_t)args.RB;
    if (nc >= (uint32_t)args.channels) return;
    const uint32_t n = fast_div(nc, args.c_mul, args.c_shift), c = nc - n * (uint32_t)a.C;
    const int oh0 = (int)rb * kRows, ow0 = (int)gc * 4, ih0 = oh0 * S - a.ph, iw0 = ow0 * S - a.pw;
    const char* plane = a.x + (int64_t)n * a.x_n_stride + (int64_t)c * a.x_c_stride;
    const uint64_t flip = a.x_signed ? 0 : 0x8080808080808080ull, zp = (uint64_t)((uint32_t)((a.x_zp_u ^ 0x80) & 0xff) * 0x01010101u) * 0x100000001ull;
    constexpr int kIn = (kRows - 1) * S + 3;
    uint64_t v[kIn], v2[kIn];  // in the signed range
#pragma unroll
    for (int r = 0; r < kIn; ++r) {
        const int ih = ih0 + r;
        const bool inside = ih >= 0 && ih < a.H;
        const char* row = plane + (int64_t)(inside ? ih : 0) * a.x_h_stride;
        if (a.W >= 8) {
            v[r] = window8(row, inside ? iw0 : a.W + 8, a.W, zp ^ flip) ^ flip;
            v2[r] = S == 2 ? window8(row, inside ? iw0 + 8 : a.W + 8, a.W, zp ^ flip) ^ flip : 0;
        } else {
            v[r] = narrow_window(row, inside ? iw0 : a.W, a.W, zp ^ flip) ^ flip;
            v2[r] = S == 2 ? narrow_window(row, inside ? iw0 + 8 : a.W, a.W, zp ^ flip) ^ flip : 0;
        }
    }
    int32_t w[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) w[i] = a.rows[(c >> 2) * 12 + i * 4 + (c & 3)];
    const int32_t bias = a.bias ? a.bias[c] : 0, seed = (128 - a.x_zp_u) * a.wsum[c] + (kFloatBias ? 0 : bias);
    const float scale = a.x_scale * (a.w_scale_len > 1 ? a.w_scale[c] : a.w_scale[0]), fb = kFloatBias ? (float)bias : 0.f;
    char* out = a.y + (int64_t)n * a.y_n_stride + (int64_t)c * a.y_c_stride + ow0;
    const int cnt = min(4, a.OW - ow0);
#pragma unroll
    for (int p = 0; p < kRows; ++p) {
        float pre[4];
        int32_t code[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            int32_t acc = seed;
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const int r = p * S + i, at = e * S;  // bytes at, at + 1, at + 2 (the fourth meets a zero)
                const uint32_t x = at == 0 ? (uint32_t)v[r] : at + 4 <= 8 ? (uint32_t)(v[r] >> (8 * at)) : (uint32_t)(v[r] >> (8 * at)) | (uint32_t)(v2[r] << (64 - 8 * at));
                acc = __builtin_amdgcn_sdot4((int)x, w[i], acc, false);
            }
            float s = (float)acc * scale;
            if (kFloatBias) s = s + fb;
            if (kPath != 0) pre[e] = quantize_prefloor_u8<kPath>(s, a.qp);
            else code[e] = rne ? quantize_value_folded<true>(s, a.q, a.inv_y_scale, a.lo_folded) : quantize_value_folded<false>(s, a.q, a.inv_y_scale, a.lo_folded);
        }
        const uint32_t o = (kPath ? floor_sat_u8x4(pre[0], pre[1], pre[2], pre[3]) : pack4(code[0], code[1], code[2], code[3])) ^ a.y_flip;
        if (oh0 + p >= a.OH) continue;
        char* dst = out + (int64_t)(oh0 + p) * a.y_h_stride;
        if (cnt == 4) *reinterpret_cast<u32_u*>(dst) = o;
        else
            for (int e = 0; e < cnt; ++e) dst[e] = (char)(o >> (8 * e));
    }
}

}  // namespace

int launch_depthwise_planar(const DepthwiseArgs& a, bool rne, hipStream_t s) {
    if (a.sh != a.sw || a.sh < 1 || a.sh > 2) return CHX_HIP_EUNSUPPORTED;
    const int G = (a.OW + 3) / 4, RB = (a.OH + kRows - 1) / kRows;
    const int64_t channels = (int64_t)a.N * a.C, total = channels * RB * G;
    if (total == 0) return CHX_HIP_OK;
    if (total >= (int64_t(1) << 31) - 256) return CHX_HIP_EUNSUPPORTED;
    DepthwisePlanarArgs args;
    args.conv = a;
    args.rne = rne ? 1 : 0;
    args.G = G;
    args.RB = RB;
    args.channels = (int32_t)channels;
    magic_divisor((uint32_t)G, &args.g_mul, &args.g_shift);
    magic_divisor((uint32_t)RB, &args.rb_mul, &args.rb_shift);
    magic_divisor((uint32_t)a.C, &args.c_mul, &args.c_shift);
    const bool fb = a.bias != nullptr && a.float_bias != 0;
    const int path = rne ? 0 : a.qp.path;
    const unsigned blocks = (unsigned)((total + 255) / 256);
#define CHX_DWP(S, P, F) depthwise_planar_kernel<S, P, F><<<blocks, 256, 0, s>>>(args)
#define CHX_DWP_F(S, P)                   \
    do {                                  \
        if (fb) CHX_DWP(S, P, true);      \
        else CHX_DWP(S, P, false);        \
    } while (0)
#define CHX_DWP_S(S)                      \
    do {                                  \
        if (path == 0) CHX_DWP_F(S, 0);   \
        else if (path == 1) CHX_DWP_F(S, 1); \
        else if (path == 2) CHX_DWP_F(S, 2); \
        else CHX_DWP_F(S, 3);             \
    } while (0)
    if (a.sh == 1) CHX_DWP_S(1);
    else CHX_DWP_S(2);
#undef CHX_DWP_S
#undef CHX_DWP_F
#undef CHX_DWP
    return launch_check("depthwise_planar_kernel");
}

}  // namespace chx
