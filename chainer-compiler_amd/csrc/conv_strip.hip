// ConvInteger in one launch: a work-group's strip of x goes into LDS once per filter column.
//
// conv_planar.hip copies x into padded planes first; for the layers of a network at a few images its two launches are 8.4
// us whatever they do.  Where the input rows of a few output rows fit LDS for all channels, that copy can stay inside the
// product's launch.  A lane multiplies four neighbouring output pixels, so for filter column kw it wants the bytes kw, kw +
// stride, ... of its input row as one dword: LDS holds that dword for every channel, filter column, input row and group of
// four output columns (sign bits flipped, padding filled in), and row k = (c, kh, kw) of the matrix is a run of aligned
// dwords at a table's offset k.  From there the product is conv_planar_kernel's: 32 filters x 128 pixels, b transposed
// in registers, K split over wavefronts, sums for the zero points.
// Bound by its serial chain: start, loads of x, two barriers, up to seven steps of K per wavefront, the sums through LDS.
// [8, 64, 56, 56] with 64 3x3 filters: 8.9 us, 14.6 with the copy in a launch of its own (channels-last 11.4 and 18.1).
#include <cstring>
#include <type_traits>

#include "contract.h"
#include "conv_mfma.h"
#include "gemm_i8_device.h"

namespace chx {
namespace {

struct StripArgs {
    const char* x;
    int64_t xs[4];
    int32_t N, C, H, W, ph, pw, KH, OH, OW;
    int32_t TR, RI, G, strips;        // output rows and input rows of a strip, groups of four output columns, strips of an image
    uint32_t zp;                      // the zero point's byte, four times, in the signed range
    const char* w;
    int64_t w_row;
    int32_t M, K;
    uint32_t w_flip, x_flip;
    int32_t cx;                       // 128 - zero point of x (or -zero point)
    const char* w_zp;
    int32_t w_zp_len, w_zp_signed;
    int64_t w_zp_stride;
    char* y;
    int64_t ys[4];
    uint32_t taps_mul, taps_shift, kw_mul, kw_shift, g_mul, g_shift, rg_mul, rg_shift;  // magic_divisor of KH * KW, KW, G, RI * G
    int32_t table_at;                 // of the offsets, behind the strip
};

__device__ __forceinline__ uint32_t divided(uint32_t n, uint32_t mul, uint32_t shift) {
    return (__umulhi(n, mul) + n) >> shift;
}

constexpr int kR = 32, kStep = 32, kRegs = 16, kWaves = 8;

// FT: filter tiles of the work-group (64 or 32 filters); its wavefronts split K kWaves / FT ways.
template <int S, int KW, bool kChannelsLast, int FT>
__global__ __launch_bounds__(64 * kWaves, 2) void conv_strip_kernel(StripArgs g) {
    constexpr int KS = kWaves / FT;
    extern __shared__ __attribute__((aligned(16))) char lds[];
    uint32_t* strip = reinterpret_cast<uint32_t*>(lds);  // [C][KW][RI][G]
    int32_t* offsets = reinterpret_cast<int32_t*>(lds + g.table_at);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane % kR, group = lane / kR;
    const int n = (int)blockIdx.x / g.strips, oh0 = ((int)blockIdx.x - n * g.strips) * g.TR;
    const int m0 = ((int)blockIdx.y * FT + wave % FT) * kR, ks = wave / FT;
    const int m_in = min(m0 + col, g.M - 1);
    const char* w_row = g.w + (int64_t)m_in * g.w_row;
    const int steps = (g.K + kStep - 1) / kStep, full = g.K / kStep;
    const int per = (steps + KS - 1) / KS, lo = ks * per, hi = min(steps, lo + per), full_hi = min(full, hi);

    // the first weights, before anything else: they come from memory
    constexpr int kDepth = 4;
    v4i fa_ring[kDepth];
    if (lo < full_hi) {
#pragma unroll
        for (int d = 0; d < kDepth; ++d) fa_ring[d] = load_k16<false>(w_row, min(lo + d, full_hi - 1) * kStep + group * 16, g.K);
    }

    // ---- the strip ----
    const int RG = g.RI * g.G;
    const char* xn = g.x + (int64_t)n * g.xs[0];
    const int ih_first = oh0 * S - g.ph;
    if constexpr (!kChannelsLast) {
        const uint64_t zp = g.zp | (uint64_t)g.zp << 32, flip = g.x_flip | (uint64_t)g.x_flip << 32;
        constexpr int kBatch = 8;  // loads in flight
        const int total = g.C * RG;
        for (int i0 = tid; i0 < total; i0 += kBatch * 64 * kWaves) {
            uint64_t v[kBatch], v2[kBatch];
            uint32_t to[kBatch];
#pragma unroll
            for (int u = 0; u < kBatch; ++u) {
                const uint32_t i = (uint32_t)min(i0 + u * 64 * kWaves, total - 1);
                const uint32_t c = divided(i, g.rg_mul, g.rg_shift), at = i - c * (uint32_t)RG;
                const uint32_t r = divided(at, g.g_mul, g.g_shift), gc = at - r * (uint32_t)g.G;
                const int ih = ih_first + (int)r, iw = (int)gc * 4 * S - g.pw;
                const bool inside = ih >= 0 && ih < g.H;
                const char* row = xn + (int64_t)c * g.xs[1] + (inside ? (int64_t)ih * g.xs[2] : 0);
                // (the fill goes through the same flip: it is given in the stored range here)
                v[u] = window8(row, inside ? iw : g.W + 8, g.W, zp ^ flip) ^ flip;
                if (S * 3 + KW > 8) v2[u] = window8(row, inside ? iw + 8 : g.W + 8, g.W, zp ^ flip) ^ flip;
                else v2[u] = 0;
                to[u] = (c * KW * (uint32_t)g.RI + r) * (uint32_t)g.G + gc;
            }
#pragma unroll
            for (int u = 0; u < kBatch; ++u) {
                if (i0 + u * 64 * kWaves >= total) break;
                uint32_t* dst = strip + to[u];
#pragma unroll
                for (int kw = 0; kw < KW; ++kw) {
                    const uint64_t s = kw == 0 ? v[u] : v[u] >> (8 * kw) | (v2[u] << (64 - 8 * kw));
                    dst[kw * RG] = S == 1 ? (uint32_t)s : __builtin_amdgcn_perm((uint32_t)(s >> 32), (uint32_t)s, 0x06040200u);
                }
            }
        }
    } else {
        constexpr int NC = 3 * S + KW;  // input columns under four output columns
        const int quads = g.C / 4;
        constexpr int kBatch = S == 1 ? 4 : 2;
        const int total = (quads + 3) / 4 * 4 * RG;
        for (int i0 = tid; i0 < total; i0 += kBatch * 64 * kWaves) {
            uint32_t v[kBatch][NC], to[kBatch];
#pragma unroll
            for (int u = 0; u < kBatch; ++u) {
                // consecutive lanes: 16 channels, then columns (more channels of a column would meet in the banks)
                const uint32_t i = (uint32_t)min(i0 + u * 64 * kWaves, total - 1);
                const uint32_t cb = divided(i >> 2, g.rg_mul, g.rg_shift), at = (i >> 2) - cb * (uint32_t)RG;
                const uint32_t cq = min(cb * 4 + (i & 3), (uint32_t)quads - 1);
                const uint32_t r = divided(at, g.g_mul, g.g_shift), gc = at - r * (uint32_t)g.G;
                const int ih = ih_first + (int)r, iw = (int)gc * 4 * S - g.pw;
                const bool inside = ih >= 0 && ih < g.H;
                const char* px = xn + (inside ? (int64_t)ih * g.xs[2] : 0) + 4 * cq;
#pragma unroll
                for (int j = 0; j < NC; ++j) {
                    const int w = min(max(iw + j, 0), g.W - 1);
                    v[u][j] = *reinterpret_cast<const u32_u*>(px + (int64_t)w * g.xs[3]) ^ g.x_flip;
                    v[u][j] = !inside || iw + j != w ? g.zp : v[u][j];
                }
                to[u] = (cq * 4 * KW * (uint32_t)g.RI + r) * (uint32_t)g.G + gc;
            }
#pragma unroll
            for (int u = 0; u < kBatch; ++u) {
                if (i0 + u * 64 * kWaves >= total) break;
                uint32_t* dst = strip + to[u];
#pragma unroll
                for (int kw = 0; kw < KW; ++kw) {
                    const uint32_t a = v[u][kw], b = v[u][kw + S], c = v[u][kw + 2 * S], d = v[u][kw + 3 * S];
                    const uint32_t t0 = __builtin_amdgcn_perm(b, a, 0x05010400u), t1 = __builtin_amdgcn_perm(b, a, 0x07030602u);
                    const uint32_t t2 = __builtin_amdgcn_perm(d, c, 0x05010400u), t3 = __builtin_amdgcn_perm(d, c, 0x07030602u);
                    dst[kw * RG] = __builtin_amdgcn_perm(t2, t0, 0x05040100u);
                    dst[(KW + kw) * RG] = __builtin_amdgcn_perm(t2, t0, 0x07060302u);
                    dst[(2 * KW + kw) * RG] = __builtin_amdgcn_perm(t3, t1, 0x05040100u);
                    dst[(3 * KW + kw) * RG] = __builtin_amdgcn_perm(t3, t1, 0x07060302u);
                }
            }
        }
    }
    // where row k of the matrix starts (in dwords); rows past K (weights 0) are read at row 0
    for (int k = tid; k < steps * kStep; k += 64 * kWaves) {
        int32_t off = 0;
        if (k < g.K) {
            const uint32_t c = divided((uint32_t)k, g.taps_mul, g.taps_shift), t = (uint32_t)k - c * (uint32_t)(g.KH * KW);
            const uint32_t kh = divided(t, g.kw_mul, g.kw_shift), kw = t - kh * (uint32_t)KW;
            off = (int32_t)(((c * KW + kw) * (uint32_t)g.RI + kh) * (uint32_t)g.G);
        }
        offsets[k] = off;
    }
    __syncthreads();

    // ---- the product (as conv_planar_kernel's) ----
    const uint32_t tr = divided((uint32_t)col, g.g_mul, g.g_shift), gc = (uint32_t)col - tr * (uint32_t)g.G;
    const bool lane_used = (int)tr < g.TR;
    const uint32_t* b = strip + (lane_used ? tr * S * (uint32_t)g.G + gc : 0u);
    auto row_of = [&](int r) { return (r / 4) * 8 + group * 4 + r % 4; };
    auto filter_c = [&](int m) -> int32_t {
        int32_t z = 0;
        if (g.w_zp) z = zero_point(g.w_zp + (g.w_zp_len > 1 ? (int64_t)min(m, g.M - 1) * g.w_zp_stride : 0), g.w_zp_signed);
        return (g.w_flip ? 128 : 0) - z;
    };
    const bool any_cw = __builtin_amdgcn_ballot_w64(filter_c(m0 + col) != 0) != 0;
    const int32_t cx = g.cx;
    v16i acc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < kRegs; ++r) acc[i][r] = 0;
    int32_t col_sum[4] = {0, 0, 0, 0}, row_sum = 0;
    auto multiply = [&](auto tail_c, int step, v4i raw) {
        constexpr bool kTail = decltype(tail_c)::value;
        const int k0 = step * kStep + group * 16;
        const v4i fa = flipped<kTail>(raw, g.w_flip, k0, g.K);
        uint32_t rows[16];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const v4i off = *reinterpret_cast<const v4i*>(&offsets[k0 + 4 * q]);
#pragma unroll
            for (int e = 0; e < 4; ++e) rows[4 * q + e] = b[off[e]];
        }
        v4i fb[4];
        transpose16x4(rows, fb);
        if (kTail && any_cw) {
            // rows past K hold bytes of row 0: they meet zero weights, but must not enter the sums
            const int left = g.K - k0;
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int keep = min(max(left - 4 * e, 0), 4);
                    fb[i][e] = keep == 4 ? fb[i][e] : fb[i][e] & (int)((1u << (8 * keep)) - 1u);
                }
        }
        if (any_cw) {
#pragma unroll
            for (int i = 0; i < 4; ++i) col_sum[i] = sum_bytes(fb[i], col_sum[i]);
        }
        if (cx != 0) row_sum = sum_bytes(fa, row_sum);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa, fb[i], acc[i], 0, 0, 0);
    };
    using no_tail = std::integral_constant<bool, false>;
    using tail = std::integral_constant<bool, true>;
    if (lo < full_hi) {
        int step = lo;
        for (; step + kDepth <= full_hi; step += kDepth) {
#pragma unroll
            for (int d = 0; d < kDepth; ++d) {
                multiply(no_tail(), step + d, fa_ring[d]);
                fa_ring[d] = load_k16<false>(w_row, min(step + d + kDepth, full_hi - 1) * kStep + group * 16, g.K);
            }
        }
#pragma unroll
        for (int d = 0; d < kDepth - 1; ++d)
            if (step + d < full_hi) multiply(no_tail(), step + d, fa_ring[d]);
    }
    if (full < steps && full >= lo && full < hi) multiply(tail(), full, load_k16<true>(w_row, full * kStep + group * 16, g.K));

    auto over_groups = [&](int32_t v) { return v + __shfl_xor(v, 32); };
    // (w' + cw)(x' + cx) summed over K: the wavefronts' shares of the sums add up like the products
    if (any_cw) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int32_t of_col = over_groups(col_sum[i]) + (ks == 0 ? g.K * cx : 0);
#pragma unroll
            for (int r = 0; r < kRegs; ++r) acc[i][r] += filter_c(m0 + row_of(r)) * of_col;
        }
    }
    if (cx != 0) {
        const int32_t mine = cx * over_groups(row_sum);
#pragma unroll
        for (int r = 0; r < kRegs; ++r) {
            const int32_t add = __shfl(mine, row_of(r));
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i][r] += add;
        }
    }

    // ---- the wavefronts' sums meet in LDS; each finishes its share of the filters ----
    const int oh = oh0 + (int)tr, ow = (int)gc * 4;
    const bool stored = lane_used && oh < g.OH;
    char* y_px = g.y + (int64_t)n * g.ys[0] + (int64_t)oh * g.ys[2] + (int64_t)ow * g.ys[3];
    const bool run = g.ys[3] == 4 && ow + 4 <= g.OW;  // one 16-byte store
    typedef int v4i_d __attribute__((ext_vector_type(4), aligned(4)));
    // (64 KB at a time: the upper four wavefronts give theirs to the lower four, which lay out what they then have)
    v4i* part = reinterpret_cast<v4i*>(lds);  // [wave % 4][register][lane]
    __syncthreads();                          // every wavefront is done with the strip
    auto give = [&]() {
#pragma unroll
        for (int r = 0; r < kRegs; ++r) part[(wave % 4 * kRegs + r) * 64 + lane] = v4i{acc[0][r], acc[1][r], acc[2][r], acc[3][r]};
    };
    if (wave >= 4) give();
    __syncthreads();
    if (wave < 4) {
#pragma unroll
        for (int r = 0; r < kRegs; ++r) {
            const v4i other = part[(wave * kRegs + r) * 64 + lane];
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i][r] += other[i];
        }
        give();  // (each its own lanes' places)
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kRegs / KS; ++i) {
        const int r = ks * (kRegs / KS) + i, m = m0 + row_of(r);
        v4i sum = part[((wave % FT) * kRegs + r) * 64 + lane];
#pragma unroll
        for (int q = 1; q < 4 / FT; ++q) sum += part[((q * FT + wave % FT) * kRegs + r) * 64 + lane];
        if (!stored || m >= g.M) continue;
        char* y = y_px + (int64_t)m * g.ys[1];
        if (run) {
            *reinterpret_cast<v4i_d*>(y) = sum;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (ow + e < g.OW) *reinterpret_cast<int32_t*>(y + (int64_t)e * g.ys[3]) = sum[e];
        }
    }
}

template <int S, int KW, bool kChannelsLast>
void launch(const StripArgs& g, size_t bytes, hipStream_t s) {
    const unsigned strips = (unsigned)(g.N * g.strips);
    if (g.M > kR) conv_strip_kernel<S, KW, kChannelsLast, 2><<<dim3(strips, (unsigned)((g.M + 2 * kR - 1) / (2 * kR))), 64 * kWaves, bytes, s>>>(g);
    else conv_strip_kernel<S, KW, kChannelsLast, 1><<<dim3(strips, 1), 64 * kWaves, bytes, s>>>(g);
}

// The strips of a call that the kernel takes, its LDS bytes, and whether x is read along its rows; false for any other call.
bool cut_strips(const ConvDirectArgs& d, StripArgs* strips, int64_t* lds, bool* along_rows) {
    const int64_t K = (int64_t)d.Cg * d.KH * d.KW;
    const bool w_dense = (d.KW == 1 || d.ws[3] == 1) && (d.KH == 1 || d.ws[2] == d.KW) && (d.Cg == 1 || d.ws[1] == d.KH * d.KW);
    if (d.requant || d.D != 1 || d.KD != 1 || d.OD != 1 || !w_dense || K < 16 || d.group != 1) return false;
    if (d.sh != d.sw || d.sh > 2 || (d.KW != 1 && d.KW != 3)) return false;
    if (d.x_signed ? (d.x_zp < -128 || d.x_zp > 127) : (d.x_zp < 0 || d.x_zp > 255)) return false;
    const bool channels_last = d.xs[1] == 1 && d.C > 1 && d.C % 4 == 0, planar = d.xs[3] == 1 && d.W >= 8;
    if (!channels_last && !planar) return false;
    StripArgs& g = *strips;
    memset(&g, 0, sizeof(g));
    // a strip is as many rows as the 32 lanes of a tile have groups of four columns for
    g.G = (d.OW + 3) / 4;
    if (g.G > 32 || d.KH > 64) return false;
    g.TR = 32 / g.G < d.OH ? 32 / g.G : d.OH;
    g.RI = (g.TR - 1) * d.sh + d.KH;
    g.strips = (d.OH + g.TR - 1) / g.TR;
    const int64_t strip = 4 * (int64_t)d.C * d.KW * g.RI * g.G, table = 4 * ((K + kStep - 1) / kStep * kStep), sums = 4 * kRegs * 1024;
    const int64_t bytes = strip + table > sums ? strip + table : sums, work_groups = (int64_t)d.N * g.strips * ((d.OC + 63) / 64);
    // Measured against the two launches (us, here / there): [8, 64, 56, 56] with 64 3x3 filters (43 KB, 224 work-groups) 8.9 /
    // 14.6, [16, 256, 28, 28] with 64 1x1 8.3 / 10.8, [4, 128, 28, 28] with 512 1x1 6.8 / 8.7; larger strips spend longer
    // filling LDS than a launch takes ([2, 128, 28, 28] with 128 3x3, 65 KB: 11.0 / 10.2), and where work-groups follow one
    // another on a compute unit it is filled once too often ([8, 64, 56, 56] with 256 1x1, 896 of them: 20.0 / 12.2).
    // Channels-last arrays cost more to bring in: not for a few work-groups (28 of them: 10.6 / 9.4).
    // Beside a long table (1024 channels of 3x3: 36 KB) a strip of that size would pass the 64 KB that any launch may ask for.
    if (strip > 48 * 1024 || bytes > 64 * 1024 || work_groups > 512 || (!planar && work_groups < 64)) return false;
    g.table_at = (int32_t)strip;
    *lds = bytes;
    *along_rows = planar;
    return true;
}

}  // namespace

bool conv_strip_takes(const ConvDirectArgs& d) {
    StripArgs g;
    int64_t bytes;
    bool planar;
    return cut_strips(d, &g, &bytes, &planar);
}

int run_conv_strip(const ConvDirectArgs& d, hipStream_t s) {
    if (d.total == 0) return CHX_HIP_OK;
    StripArgs g;
    int64_t bytes;
    bool planar;
    if (!cut_strips(d, &g, &bytes, &planar)) return CHX_HIP_EUNSUPPORTED;
    g.x = d.x; g.w = d.w; g.y = d.y;
    for (int i = 0; i < 4; ++i) {
        g.xs[i] = d.xs[i];
        g.ys[i] = d.ys[i];
    }
    g.N = d.N; g.C = d.C; g.H = d.H; g.W = d.W; g.ph = d.ph; g.pw = d.pw; g.KH = d.KH; g.OH = d.OH; g.OW = d.OW;
    g.x_flip = d.x_signed ? 0u : 0x80808080u;
    g.w_flip = d.w_signed ? 0u : 0x80808080u;
    g.zp = (((uint32_t)d.x_zp & 0xffu) * 0x01010101u) ^ g.x_flip;
    g.cx = (d.x_signed ? 0 : 128) - d.x_zp;
    g.w_row = d.ws[0]; g.M = d.OC; g.K = (int32_t)((int64_t)d.Cg * d.KH * d.KW);
    g.w_zp = d.w_zp_len ? d.w_zp : nullptr; g.w_zp_len = d.w_zp_len; g.w_zp_stride = d.w_zp_stride; g.w_zp_signed = d.w_signed;
    magic_divisor((uint32_t)(d.KH * d.KW), &g.taps_mul, &g.taps_shift);
    magic_divisor((uint32_t)d.KW, &g.kw_mul, &g.kw_shift);
    magic_divisor((uint32_t)g.G, &g.g_mul, &g.g_shift);
    magic_divisor((uint32_t)(g.RI * g.G), &g.rg_mul, &g.rg_shift);
#define CHX_STRIP(S, KW_)                                              \
    if (d.sh == S && d.KW == KW_) {                                    \
        if (planar) launch<S, KW_, false>(g, (size_t)bytes, s);        \
        else launch<S, KW_, true>(g, (size_t)bytes, s);                \
    }
    CHX_STRIP(1, 1)
    CHX_STRIP(1, 3)
    CHX_STRIP(2, 1)
    CHX_STRIP(2, 3)
#undef CHX_STRIP
    return launch_check("conv_strip_kernel");
}

}  // namespace chx
