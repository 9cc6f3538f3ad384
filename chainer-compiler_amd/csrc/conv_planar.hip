// ConvInteger without packed weights: a matrix product that finds the convolution's rows in a padded copy of x.
//
// A call of ConvInteger brings its weights along, so nothing can be prepared before it.  Two launches:
//   1. x is copied into planes that contain the padding (bytes of the zero point), whatever its layout; with a stride s
//      the pixels of each of the s*s phases lie together.  In these planes the input of filter tap (kh, kw) of
//      neighbouring output pixels is neighbouring bytes, at a distance that depends on the tap only.
//   2. weights [OC, K = C*KH*KW] as they are  x  matrix [K, pixels] whose row k starts at a table's offset k: the product
//      of gemm_i8.hip (b's rows transposed in registers, K split over wavefronts).  Pixels run through the whole padded
//      planes, all images in a row; those that are no output pixels (the padding columns and rows: (W+1)(H+1) / WH of
//      the work for a 3x3 filter with padding 1) are computed and not stored.  Padding between neighbouring rows and
//      images is shared: one column serves as the right border of a row and the left one of the next.
// Zero points of the weights, per channel too, come in through the sums of x (see gemm_i8.hip).
//
// [8, 64, 56, 56] with 64 3x3 filters, NCHW: 1706 us with one thread per result; the copy 4.4 us and the product 10.7
// here, bound by its serial chain of loads (18 steps of K over 4 wavefronts).  Channels-last arrays: 18.5 us per call,
// against 73 with the packed kernel (conv_mfma), which needs a read-back of the zero points, three allocations and a
// packing launch per call.
#include <cstring>
#include <type_traits>

#include "contract.h"
#include "conv_mfma.h"
#include "gemm_i8_device.h"

namespace chx {
namespace {

struct PlanarArgs {
    // x [N, C, H, W] in any layout -> planes [C][s*s phases][N][Hq][Wq]
    const char* x;
    int64_t xs[4];
    char* planes;
    int32_t N, C, H, W, s_h, s_w, ph, pw, Hq, Wq;
    int64_t phase_bytes, chan_bytes;  // the images of a phase and some rows of padding; the phases of a channel and the slack behind them
    int32_t plane_rows;               // padded rows of a channel over all phases: s_h * (N * Hq + the rows of padding)
    uint32_t zp;                      // the zero point's byte, four times
    // the product
    const char* w;
    int64_t w_row;
    int32_t M, K, KH, KW, taps, P;    // P: pixels in the planes, N * Hq * Wq
    int32_t OH, OW;
    uint32_t w_flip, x_flip;
    int32_t cx;                       // 128 - zero point of x (or -zero point)
    const char* w_zp;
    int32_t w_zp_len, w_zp_signed;
    int64_t w_zp_stride;
    char* y;
    int64_t ys[4];
    int32_t group, tiles_m, tiles, tiles_per_xcd;
    uint32_t wq_mul, wq_shift, hq_mul, hq_shift, taps_mul, taps_shift, kw_mul, kw_shift, words_mul, words_shift;
};

__device__ __forceinline__ uint32_t divided(uint32_t n, uint32_t mul, uint32_t shift) {
    return (__umulhi(n, mul) + n) >> shift;
}

constexpr int kMostK = 12288, kMostTable = 4 * (kMostK + 64);
constexpr int kTileW = 64, kTileC = 64;

// Padded row `row` of a channel (rows of all images and of the padding behind them): where it comes from, and where its
// phases start in the planes.
struct PlaneRow {
    bool inside;
    int32_t n, h;
    int64_t dst;
};
__device__ __forceinline__ PlaneRow plane_row(const PlanarArgs& a, int row) {
    const uint32_t q = (uint32_t)row / (uint32_t)a.s_h, f = (uint32_t)row - q * (uint32_t)a.s_h;
    const uint32_t n = divided(q, a.hq_mul, a.hq_shift), qh = q - n * (uint32_t)a.Hq;
    PlaneRow r;
    r.n = (int32_t)n;
    r.h = (int32_t)(qh * (uint32_t)a.s_h + f) - a.ph;
    r.inside = r.n < a.N && r.h >= 0 && r.h < a.H;
    r.dst = (int64_t)f * a.s_w * a.phase_bytes + (int64_t)q * a.Wq;
    return r;
}

__device__ __forceinline__ void store_bytes(char* p, uint32_t v, int n) {
    if (n >= 4) *reinterpret_cast<u32_u*>(p) = v;
    else
        for (int i = 0; i < n; ++i) p[i] = (char)(v >> (8 * i));
}

// x with its columns running fastest (or in any other layout): a thread writes four bytes of each phase of a row.
// 4.4 us for 1.6 MB (6.8 with single bytes through LDS).
__global__ __launch_bounds__(256) void planes_kernel(PlanarArgs a) {
    const int words = (a.Wq + 3) / 4;
    const uint32_t idx = blockIdx.x * 256u + threadIdx.x;
    const uint32_t row = divided(idx, a.words_mul, a.words_shift);
    if (row >= (uint32_t)a.plane_rows) return;
    const int j = (int)(idx - row * (uint32_t)words), c = blockIdx.y;
    const PlaneRow pr = plane_row(a, (int)row);
    const int span = 4 * a.s_w, iw = j * span - a.pw;
    uint32_t lo = a.zp, hi = a.zp;
    if (pr.inside) {
        const char* src = a.x + (int64_t)pr.n * a.xs[0] + (int64_t)c * a.xs[1] + (int64_t)pr.h * a.xs[2];
        if (a.xs[3] == 1 && iw >= 0 && iw + span <= a.W) {
            lo = *reinterpret_cast<const u32_u*>(src + iw);
            if (span == 8) hi = *reinterpret_cast<const u32_u*>(src + iw + 4);
        } else {
            for (int i = 0; i < span; ++i) {
                const int at = iw + i;
                if (at < 0 || at >= a.W) continue;
                const uint32_t v = *reinterpret_cast<const uint8_t*>(src + (int64_t)at * a.xs[3]);
                uint32_t& to = i < 4 ? lo : hi;
                to = (to & ~(0xffu << (8 * (i & 3)))) | v << (8 * (i & 3));
            }
        }
    }
    char* dst = a.planes + (int64_t)c * a.chan_bytes + pr.dst + 4 * j;
    const int n = a.Wq - 4 * j;
    if (span == 4) {
        store_bytes(dst, lo, n);
    } else {
        store_bytes(dst, __builtin_amdgcn_perm(hi, lo, 0x06040200u), n);
        store_bytes(dst + a.phase_bytes, __builtin_amdgcn_perm(hi, lo, 0x07050301u), n);
    }
}

// x with its channels running fastest: 64 columns x 64 channels of a row through LDS.
__global__ __launch_bounds__(256) void planes_channels_last_kernel(PlanarArgs a) {
    __shared__ __attribute__((aligned(16))) uint8_t tile[kTileW][kTileC + 4];
    const int c0 = blockIdx.z * kTileC, w0 = blockIdx.x * kTileW;
    const int cn = min(kTileC, a.C - c0), wn = min(kTileW, a.Wq * a.s_w - w0);
    const PlaneRow pr = plane_row(a, blockIdx.y);
    const char* src = a.x + (pr.inside ? (int64_t)pr.n * a.xs[0] + (int64_t)pr.h * a.xs[2] + c0 : 0);
    const int c4 = threadIdx.x & 15;
#pragma unroll
    for (int i = 0; i < kTileW / 16; ++i) {
        const int w = (threadIdx.x >> 4) + 16 * i, iw = w0 + w - a.pw;
        uint32_t v = a.zp;
        if (pr.inside && w < wn && iw >= 0 && iw < a.W) {
            const char* p = src + (int64_t)iw * a.xs[3] + 4 * c4;
            if (4 * c4 + 4 <= cn) {
                v = *reinterpret_cast<const u32_u*>(p);
            } else {
                v = 0;
                for (int e = 0; e < 3; ++e)
                    if (4 * c4 + e < cn) v |= (uint32_t) * reinterpret_cast<const uint8_t*>(p + e) << (8 * e);
            }
        }
        *reinterpret_cast<uint32_t*>(&tile[w][4 * c4]) = v;
    }
    __syncthreads();
    // lane: a channel; four columns of one phase per step
    const int c = threadIdx.x & 63;
    if (c >= cn) return;
    const int qn = wn / a.s_w;  // columns per phase (w0 and wn are multiples of s_w)
    char* dst = a.planes + (int64_t)(c0 + c) * a.chan_bytes + pr.dst + w0 / a.s_w;
    for (int g = threadIdx.x >> 6; g < 16; g += 4) {
        const int phase = a.s_w == 2 ? g >> 3 : 0, w = 4 * (a.s_w == 2 ? g & 7 : g);
        if (w >= qn) continue;
        uint32_t v = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) v |= (uint32_t)tile[min((w + e) * a.s_w + phase, kTileW - 1)][c] << (8 * e);
        store_bytes(dst + (int64_t)phase * a.phase_bytes + w, v, qn - w);
    }
}

// Tile of R filters x 4R pixels per work-group; W wavefronts share K out (see gemm_i8_split_kernel; for the launch
// bounds conv_stem_kernel).
template <int R, int W>
__global__ __launch_bounds__(64 * W, 2) void conv_planar_kernel(PlanarArgs g) {
    constexpr int kGroups = 64 / R, kStep = 16 * kGroups, kRegs = R * R / 64, kDepth = 2;
    using acc_t = typename std::conditional<R == 32, v16i, v4i>::type;
    // the offsets of K (rounded up to a step), later the partial sums [W][kRegs][64]; large sums as a static array, the
    // launch otherwise sizes it
    constexpr int kSums = W * kRegs * 1024;
    extern __shared__ __attribute__((aligned(16))) char lds_sized[];
    __shared__ __attribute__((aligned(16))) char lds_static[kSums >= kMostTable ? kSums : 16];
    char* lds = kSums >= kMostTable ? lds_static : lds_sized;
    int32_t* offsets = reinterpret_cast<int32_t*>(lds);
    v4i* part = reinterpret_cast<v4i*>(lds);
    const int tile = (int)(blockIdx.x & 7) * g.tiles_per_xcd + (int)(blockIdx.x >> 3);
    if (tile >= g.tiles || (int)(blockIdx.x >> 3) >= g.tiles_per_xcd) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane % R, group = lane / R;
    const int m0 = (tile % g.tiles_m) * R, p0 = (tile / g.tiles_m) * 4 * R;
    const int grp = blockIdx.y;  // of the convolution

    // where row k of the matrix starts; rows past K (weights 0) are read at row 0
    const int steps = (g.K + kStep - 1) / kStep;
    for (int k = threadIdx.x; k < steps * kStep; k += 64 * W) {
        int32_t off = 0;
        if (k < g.K) {
            const uint32_t c = divided((uint32_t)k, g.taps_mul, g.taps_shift), t = (uint32_t)k - c * (uint32_t)g.taps;
            const uint32_t kh = divided(t, g.kw_mul, g.kw_shift), kw = t - kh * (uint32_t)g.KW;
            const uint32_t fh = kh % (uint32_t)g.s_h, fw = kw % (uint32_t)g.s_w;
            off = (int32_t)(c * (uint32_t)g.chan_bytes + (fh * (uint32_t)g.s_w + fw) * (uint32_t)g.phase_bytes + kh / (uint32_t)g.s_h * (uint32_t)g.Wq + kw / (uint32_t)g.s_w);
        }
        offsets[k] = off;
    }
    __syncthreads();

    const char* planes = g.planes + (int64_t)grp * (g.C / g.group) * g.chan_bytes;
    const int p = p0 + 4 * col;  // the lane's four pixels (past the last one: bytes of the slack or of other planes)
    const uint32_t voff = (uint32_t)min(p, g.P - 1);
    const int m_in = min(m0 + col, g.M - 1);
    const char* w_row = g.w + ((int64_t)grp * g.M + m_in) * g.w_row;

    // zero points of the filters of this lane's result rows (and whether any filter of the tile has one)
    auto row_of = [&](int r) { return (r / 4) * (4 * kGroups) + group * 4 + r % 4; };
    auto filter_c = [&](int m) -> int32_t {
        int32_t z = 0;
        if (g.w_zp) z = zero_point(g.w_zp + (g.w_zp_len > 1 ? ((int64_t)grp * g.M + min(m, g.M - 1)) * g.w_zp_stride : 0), g.w_zp_signed);
        return (g.w_flip ? 128 : 0) - z;
    };
    const bool any_cw = __builtin_amdgcn_ballot_w64(filter_c(m0 + col) != 0) != 0;
    const int32_t cx = g.cx;

    acc_t acc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < kRegs; ++r) acc[i][r] = 0;
    int32_t col_sum[4] = {0, 0, 0, 0}, row_sum = 0;

    struct Step {
        v4i fa;
        uint32_t w[16];
    };
    auto load = [&](auto tail_c, int step, Step& s) {
        constexpr bool kTail = decltype(tail_c)::value;
        const int k0 = step * kStep + group * 16;
        s.fa = load_k16<kTail>(w_row, k0, g.K);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const v4i off = *reinterpret_cast<const v4i*>(&offsets[k0 + 4 * q]);
#pragma unroll
            for (int e = 0; e < 4; ++e) s.w[4 * q + e] = *reinterpret_cast<const u32_u*>(planes + (uint32_t)((uint32_t)off[e] + voff));
        }
    };
    auto multiply = [&](auto tail_c, int step, Step& s) {
        constexpr bool kTail = decltype(tail_c)::value;
        const int k0 = step * kStep + group * 16;
        const v4i fa = flipped<kTail>(s.fa, g.w_flip, k0, g.K);
        v4i fb[4];
        columns_of<false>(s.w, false, 0, g.x_flip, 0, 0, fb);
        if (kTail && any_cw) {
            // rows past K hold bytes of row 0: they meet zero weights, but must not enter the sums
            const int left = g.K - k0;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (left <= 0) fb[i] = v4i{0, 0, 0, 0};
                else if (left < 16) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int keep = min(max(left - 4 * e, 0), 4);
                        fb[i][e] = keep == 4 ? fb[i][e] : fb[i][e] & (int)((1u << (8 * keep)) - 1u);
                    }
                }
            }
        }
        if (any_cw) {
#pragma unroll
            for (int i = 0; i < 4; ++i) col_sum[i] = sum_bytes(fb[i], col_sum[i]);
        }
        if (cx != 0) row_sum = sum_bytes(fa, row_sum);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (R == 32) acc[i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa, fb[i], acc[i], 0, 0, 0);
            else acc[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa, fb[i], acc[i], 0, 0, 0);
        }
    };
    const int full = g.K / kStep, per = (steps + W - 1) / W, lo = wave * per, hi = min(steps, lo + per), full_hi = min(full, hi);
    using no_tail = std::integral_constant<bool, false>;
    using tail = std::integral_constant<bool, true>;
    if (lo < full_hi) {
        Step ring[kDepth];
#pragma unroll
        for (int d = 0; d < kDepth; ++d) load(no_tail(), min(lo + d, full_hi - 1), ring[d]);
        int step = lo;
        for (; step + kDepth <= full_hi; step += kDepth) {
#pragma unroll
            for (int d = 0; d < kDepth; ++d) {
                multiply(no_tail(), 0, ring[d]);
                load(no_tail(), min(step + d + kDepth, full_hi - 1), ring[d]);
            }
        }
#pragma unroll
        for (int d = 0; d < kDepth - 1; ++d)
            if (step + d < full_hi) multiply(no_tail(), 0, ring[d]);
    }
    if (full < steps && full >= lo && full < hi) {
        Step last;
        load(tail(), full, last);
        multiply(tail(), full, last);
    }

    auto over_groups = [&](int32_t v) {
        if (R == 16) v += __shfl_xor(v, 16);
        return v + __shfl_xor(v, 32);
    };
    // (w' + cw)(x' + cx) summed over K: the wavefronts' shares of the sums add up like the products
    if (any_cw) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int32_t of_col = over_groups(col_sum[i]) + (wave == 0 ? g.K * cx : 0);
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

    // where the lane's four pixels go, -1: not an output pixel
    int64_t at[4];
    {
        uint32_t row = divided((uint32_t)min(p, g.P - 1), g.wq_mul, g.wq_shift);
        uint32_t ow = (uint32_t)min(p, g.P - 1) - row * (uint32_t)g.Wq;
        uint32_t img = divided(row, g.hq_mul, g.hq_shift), oh = row - img * (uint32_t)g.Hq;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            at[i] = p + i < g.P && ow < (uint32_t)g.OW && oh < (uint32_t)g.OH ? (int64_t)img * g.ys[0] + (int64_t)oh * g.ys[2] + (int64_t)ow * g.ys[3] : -1;
            if (++ow == (uint32_t)g.Wq) {
                ow = 0;
                if (++oh == (uint32_t)g.Hq) oh = 0, ++img;
            }
        }
    }
    const bool run = at[0] >= 0 && at[3] >= 0 && at[3] - at[0] == 12 && at[1] - at[0] == 4 && at[2] - at[0] == 8;  // one 16-byte store
    typedef int v4i_d __attribute__((ext_vector_type(4), aligned(4)));
    auto store = [&](int m, v4i v) {
        if (m >= g.M) return;
        char* y = g.y + ((int64_t)grp * g.M + m) * g.ys[1];
        if (run) {
            *reinterpret_cast<v4i_d*>(y + at[0]) = v;
            return;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (at[i] >= 0) *reinterpret_cast<int32_t*>(y + at[i]) = v[i];
    };
    if constexpr (W == 1) {
#pragma unroll
        for (int r = 0; r < kRegs; ++r) store(m0 + row_of(r), v4i{acc[0][r], acc[1][r], acc[2][r], acc[3][r]});
    } else {
        __syncthreads();  // every wavefront is done with the offsets
#pragma unroll
        for (int r = 0; r < kRegs; ++r) part[(wave * kRegs + r) * 64 + lane] = v4i{acc[0][r], acc[1][r], acc[2][r], acc[3][r]};
        __syncthreads();
#pragma unroll
        for (int r0 = 0; r0 < kRegs; r0 += W) {
            const int r = r0 + wave;
            if (r >= kRegs) break;
            v4i sum = part[r * 64 + lane];
#pragma unroll
            for (int w = 1; w < W; ++w) sum += part[(w * kRegs + r) * 64 + lane];
            store(m0 + row_of(r), sum);
        }
    }
}

template <int R, int W>
void launch_product(const PlanarArgs& g, hipStream_t s) {
    constexpr int kRegs = R * R / 64, kStep = 16 * (64 / R);
    const size_t table = sizeof(int32_t) * (size_t)((g.K + kStep - 1) / kStep * kStep), sums = W > 1 ? (size_t)W * kRegs * 1024 : 0;
    const size_t sized = sums >= (size_t)kMostTable ? 0 : table > sums ? table : sums;
    conv_planar_kernel<R, W><<<dim3((unsigned)(8 * g.tiles_per_xcd), (unsigned)g.group), 64 * W, sized, s>>>(g);
}

}  // namespace

int run_conv_planar(const ConvDirectArgs& d, hipStream_t s) {
    if (d.total == 0) return CHX_HIP_OK;
    const int64_t K = (int64_t)d.Cg * d.KH * d.KW;
    const bool w_dense = (d.KW == 1 || d.ws[3] == 1) && (d.KH == 1 || d.ws[2] == d.KW) && (d.Cg == 1 || d.ws[1] == d.KH * d.KW);
    // the table of K offsets lies in LDS; 16 bytes of every filter are read at once
    if (d.requant || d.D != 1 || d.KD != 1 || d.OD != 1 || !w_dense || K < 16 || K > kMostK || d.group > 65535) return CHX_HIP_EUNSUPPORTED;
    if (d.sh > 2 || d.sw > 2 || d.sh < 1 || d.sw < 1) return CHX_HIP_EUNSUPPORTED;
    PlanarArgs g;
    memset(&g, 0, sizeof(g));
    g.x = d.x; g.w = d.w; g.y = d.y;
    for (int i = 0; i < 4; ++i) {
        g.xs[i] = d.xs[i];
        g.ys[i] = d.ys[i];
    }
    g.N = d.N; g.C = d.C; g.H = d.H; g.W = d.W; g.s_h = d.sh; g.s_w = d.sw; g.ph = d.ph; g.pw = d.pw;
    // padded extents: the data behind its begin padding, and room for the last window, whose end may lie in the begin
    // padding of the next row (image)
    auto padded = [](int64_t in, int64_t pad, int64_t out, int64_t k, int64_t stride) {
        const int64_t a = pad + in, b = (out - 1) * stride + k - pad;
        const int64_t q = ((a > b ? a : b) + stride - 1) / stride;
        return q > out ? q : out;  // (a place of its own for every output pixel)
    };
    const int64_t Hq = padded(d.H, d.ph, d.OH, d.KH, d.sh), Wq = padded(d.W, d.pw, d.OW, d.KW, d.sw), P = (int64_t)d.N * Hq * Wq;
    // behind the last image the begin padding that its last windows share with a next one; behind a channel room for
    // the windows of pixels that are no output pixels, whatever bytes they hold
    const int64_t extra = (d.ph + d.sh - 1) / d.sh + 1, phase = ((int64_t)d.N * Hq + extra) * Wq;
    const int64_t slack = ((int64_t)d.KH * Wq + d.KW + 64 + 63) / 64 * 64;
    const int64_t chan = d.sh * d.sw * phase + slack, bytes = chan * d.C, plane_rows = d.sh * ((int64_t)d.N * Hq + extra);
    if (bytes >= (int64_t(1) << 31) || plane_rows > 65535 || d.C > 65535 || plane_rows * ((Wq + 3) / 4) >= (int64_t(1) << 31) - 256) return CHX_HIP_EUNSUPPORTED;
    g.Hq = (int32_t)Hq; g.Wq = (int32_t)Wq; g.P = (int32_t)P;
    g.phase_bytes = phase; g.chan_bytes = chan; g.plane_rows = (int32_t)plane_rows;
    const uint32_t zp = (uint32_t)d.x_zp & 0xffu;
    g.zp = zp * 0x01010101u;
    g.w_row = d.ws[0];
    g.M = d.OC / d.group; g.K = (int32_t)K; g.KH = d.KH; g.KW = d.KW; g.taps = d.KH * d.KW;
    g.OH = d.OH; g.OW = d.OW; g.group = d.group;
    g.x_flip = d.x_signed ? 0u : 0x80808080u;
    g.w_flip = d.w_signed ? 0u : 0x80808080u;
    g.cx = (d.x_signed ? 0 : 128) - d.x_zp;
    // the padding holds the zero point as a byte of x's type
    if (d.x_signed ? (d.x_zp < -128 || d.x_zp > 127) : (d.x_zp < 0 || d.x_zp > 255)) return CHX_HIP_EUNSUPPORTED;
    g.w_zp = d.w_zp_len ? d.w_zp : nullptr; g.w_zp_len = d.w_zp_len; g.w_zp_stride = d.w_zp_stride; g.w_zp_signed = d.w_signed;
    magic_divisor((uint32_t)Wq, &g.wq_mul, &g.wq_shift);
    magic_divisor((uint32_t)Hq, &g.hq_mul, &g.hq_shift);
    magic_divisor((uint32_t)g.taps, &g.taps_mul, &g.taps_shift);
    magic_divisor((uint32_t)d.KW, &g.kw_mul, &g.kw_shift);
    Scratch scratch;
    CHX_PROPAGATE(scratch.acquire((size_t)bytes, s));
    g.planes = static_cast<char*>(scratch.ptr());
    const int64_t words = (Wq + 3) / 4;
    magic_divisor((uint32_t)words, &g.words_mul, &g.words_shift);
    if (d.xs[1] == 1 && d.C > 1) {
        const dim3 grid((unsigned)((Wq * d.sw + kTileW - 1) / kTileW), (unsigned)plane_rows, (unsigned)((d.C + kTileC - 1) / kTileC));
        planes_channels_last_kernel<<<grid, 256, 0, s>>>(g);
    } else {
        planes_kernel<<<dim3((unsigned)((plane_rows * words + 255) / 256), (unsigned)d.C), 256, 0, s>>>(g);
    }
    CHX_PROPAGATE(launch_check("planes_kernel"));
    auto tiles = [&](int tm, int tp) {
        g.tiles_m = (g.M + tm - 1) / tm;
        const int64_t t = (int64_t)g.tiles_m * ((P + tp - 1) / tp);
        g.tiles = (int32_t)t;
        g.tiles_per_xcd = (int32_t)((t + 7) / 8);
        return t;
    };
    // tile and split as for the plain product (launch_matmul_i8)
    const bool small = g.M <= 16 || tiles(32, 128) * d.group <= 128;
    const int64_t work_groups = tiles(small ? 16 : 32, small ? 64 : 128) * d.group, steps = (K + (small ? 63 : 31)) / (small ? 64 : 32);
    int w = 1;
    while (w < 8 && 2 * w <= steps && 2 * w * work_groups <= 2048) w *= 2;
    if (small) {
        if (w == 1) launch_product<16, 1>(g, s);
        else if (w == 2) launch_product<16, 2>(g, s);
        else if (w == 4) launch_product<16, 4>(g, s);
        else launch_product<16, 8>(g, s);
    } else {
        if (w == 1) launch_product<32, 1>(g, s);
        else if (w == 2) launch_product<32, 2>(g, s);
        else if (w == 4) launch_product<32, 4>(g, s);
        else launch_product<32, 8>(g, s);
    }
    return launch_check("conv_planar_kernel");
}

}  // namespace chx
