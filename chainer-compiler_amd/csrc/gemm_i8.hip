// Integer matrix products on the int8 matrix cores: MatMulInteger and QLinearMatMul.
//
//   y[m, n] = sum_k (a[m, k] - za) * (b[k, n] - zb[n])      exact int32; then the int32 itself, or the requantized code
//
// Both operands are read as they are: nothing is packed, expanded or copied first, no scratch memory, no value that
// the host has to read back (the zero points are fetched by the kernel), so a call is one launch, also inside a
// recorded run.  (Packing b for the convolution kernel cost 22 us beside a product of 18 us for [1024, 1024] x [1024, 4096].)
//
// Fragments.  v_mfma_i32_32x32x32_i8 wants 16 consecutive k of one row (column) per lane.  A row of a has them in
// memory.  b is [K, N] with n running fastest: a lane reads 16 rows of 4 neighbouring columns (16 dwords) and
// transposes 4x4 byte blocks in registers (32 v_perm for 64 bytes); it then holds 16 k of columns 4j .. 4j+3, which
// serve four MFMAs, MFMA i taking column 4j+i as its column j.  The permutation of columns costs nothing: the result
// comes out with four neighbouring columns per lane, which is one 16-byte (int32) or 4-byte (code) store.
//
// Unsigned operands are made signed by flipping the top bit (a - 128); what is left of the zero points,
// ca = 128 - za (or -za) and cb[n], enters through the sums of the other operand:
//   sum (a' + ca)(b' + cb) = sum a'b' + ca * sum_k b' + cb * sum_k a' + K ca cb
// The sums are dot products with ones on the fragments that are in registers anyway, taken only when ca (cb) is not 0.
//
// Rows of any length and alignment: a group of 16 k that reaches past K is read as the last 16 bytes of its row and
// shifted down (zeros move in), and likewise a dword that reaches past N as the last 4 bytes, so no access leaves a row.
#include <cmath>
#include <cstring>
#include <type_traits>

#include "contract.h"
#include "gemm_i8_device.h"

namespace chx {
namespace {

struct GemmI8Args {
    const char* a;
    const char* b;
    char* y;
    int64_t a_batch, a_row, b_batch, b_ld, y_batch, y_row;  // bytes; b_ld: from one k to the next, or (b transposed) from one n to the next
    int32_t M, N, K;
    uint32_t a_flip, b_flip;  // 0x80808080 for an unsigned operand
    const char* a_zp;         // one element, or null: a_zp_imm
    const char* b_zp;         // b_zp_len elements, or null: b_zp_imm
    int32_t b_zp_len;
    int64_t b_zp_stride;
    int32_t a_zp_signed, b_zp_signed, a_zp_imm, b_zp_imm;
    int32_t tiles_m, tiles, tiles_per_xcd;
    // epilogue
    int32_t requant, rne;
    int32_t finish;       // Finish
    float b_scale;
    const int32_t* bias;
    RequantParams rq;
    float inv_y_scale, lo_folded;  // for kFolded*
    QuantProduct qp;               // for kProduct*
};

// How a sum becomes a code.  kProduct + path and the folded forms give the codes of the exact ones (quant_math.h) wherever
// no intermediate value leaves the range of float32, which the launcher checks; the exact ones divide, about twice the
// instructions: QLinearMatMul of 8192 x 256 x 8192, whose results are many for its products, 113 us with them and 60 without.
enum Finish : int32_t { kFolded = 0, kProduct1 = 1, kProduct2 = 2, kProduct3 = 3, kFoldedRne = 4, kExact = 5 };

// Four neighbouring int32 results n .. n+3 of one row.
__device__ __forceinline__ void store4(const GemmI8Args& g, char* y, int m, int n, v4i acc) {
    if (m >= g.M || n >= g.N) return;
    typedef int v4i_d __attribute__((ext_vector_type(4), aligned(4)));
    int32_t* p = reinterpret_cast<int32_t*>(y + (int64_t)m * g.y_row) + n;
    if (n + 4 <= g.N) __builtin_nontemporal_store(acc, reinterpret_cast<v4i_d*>(p));
    else
        for (int i = 0; i < 3; ++i)
            if (n + i < g.N) p[i] = acc[i];
}

// The codes of such results in kRows (1, 2 or 4) rows m[..].
template <int kFinish, int kRows>
__device__ __forceinline__ void store_codes(const GemmI8Args& g, char* y, const int (&m)[kRows], int n, const v4i (&acc)[kRows], v4i bias) {
    uint32_t word[kRows];
    const float s = g.rq.x_scale * g.b_scale;
    if constexpr (kFinish == kProduct1 || kFinish == kProduct2 || kFinish == kProduct3) {
        float pre[4 * kRows];
#pragma unroll
        for (int r = 0; r < kRows; ++r)
#pragma unroll
            for (int i = 0; i < 4; ++i) pre[4 * r + i] = quantize_prefloor_u8<kFinish>((float)(acc[r][i] + bias[i]) * s, g.qp);
        if constexpr (kRows == 4) floor_sat_u8x16(pre, word);
        else if constexpr (kRows == 2) floor_sat_u8x8(pre, &word[0], &word[1]);
        else word[0] = floor_sat_u8x4(pre[0], pre[1], pre[2], pre[3]);
    } else {
#pragma unroll
        for (int r = 0; r < kRows; ++r) {
            int32_t code[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int32_t v = acc[r][i] + bias[i];
                if constexpr (kFinish == kFolded) code[i] = quantize_value_folded<false>((float)v * s, g.rq.q, g.inv_y_scale, g.lo_folded);
                else if constexpr (kFinish == kFoldedRne) code[i] = quantize_value_folded<true>((float)v * s, g.rq.q, g.inv_y_scale, g.lo_folded);
                else code[i] = g.rne ? requantize_value<true>(v, g.b_scale, 0, g.rq) : requantize_value<false>(v, g.b_scale, 0, g.rq);
            }
            word[r] = pack4(code[0], code[1], code[2], code[3]);
        }
    }
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
        if (m[r] >= g.M || n >= g.N) continue;
        uint8_t* p = reinterpret_cast<uint8_t*>(y + (int64_t)m[r] * g.y_row) + n;
        if (n + 4 <= g.N) *reinterpret_cast<u32_u*>(p) = word[r];
        else
            for (int i = 0; i < 3; ++i)
                if (n + i < g.N) p[i] = (uint8_t)(word[r] >> (8 * i));
    }
}

// A lane's results in kCount rows: sum(i) gives the four of row(i), for i < count (the same in every lane).
template <int kCount, class Row, class Sum>
__device__ __forceinline__ void store_all(const GemmI8Args& g, char* y, int n, int count, Row row, Sum sum) {
    if (!g.requant) {
#pragma unroll
        for (int i = 0; i < kCount; ++i)
            if (i < count) store4(g, y, row(i), n, sum(i));
        return;
    }
    v4i bias = {0, 0, 0, 0};  // (the ONNX kind: added to the sum)
    if (g.bias) {
#pragma unroll
        for (int i = 0; i < 4; ++i) bias[i] = g.bias[n + i < g.N ? n + i : g.N - 1];
    }
    auto finish = [&](auto how) {
        constexpr int kRows = kCount % 4 == 0 ? 4 : kCount % 2 == 0 ? 2 : 1;
#pragma unroll
        for (int i = 0; i < kCount; i += kRows) {
            if (i < count) {
                int m[kRows];
                v4i acc[kRows];
#pragma unroll
                for (int r = 0; r < kRows; ++r) {
                    m[r] = row(i + r);
                    acc[r] = sum(i + r);
                }
                store_codes<decltype(how)::value, kRows>(g, y, m, n, acc, bias);
            }
        }
    };
    switch (g.finish) {
        case kProduct1: return finish(std::integral_constant<int, kProduct1>());
        case kProduct2: return finish(std::integral_constant<int, kProduct2>());
        case kProduct3: return finish(std::integral_constant<int, kProduct3>());
        case kFolded: return finish(std::integral_constant<int, kFolded>());
        case kFoldedRne: return finish(std::integral_constant<int, kFoldedRne>());
        default: return finish(std::integral_constant<int, kExact>());
    }
}

// Work-groups go round-robin over the 8 XCDs: each XCD takes a contiguous run of tiles, m fastest, so the work-groups
// that read the same columns of b find them in one L2.
__device__ __forceinline__ int tile_of_block(const GemmI8Args& g) {
    return (int)(blockIdx.x & 7) * g.tiles_per_xcd + (int)(blockIdx.x >> 3);
}

// Tile of R rows x 4R columns per work-group (R = 16 or 32); its W wavefronts share K out and add their sums through LDS at the end.
// No LDS on the way in: a wavefront's fragments come straight from memory, three K steps ahead in registers.  Bound by
// latency (a step costs about a microsecond when nothing hides it, so K is split and the loads run ahead) and, with many
// tiles, by the vector instructions of the transposition.  One thread per result, K serial, took 160 us for
// 197 x 770 x 1001; this 6.0.  1024 x 1024 x 4096: 14 us, against 22 us of packing and 18 us on the convolution kernel.
// (Launch bounds: see conv_stem_kernel.)
template <int R, int W, bool kBT, bool kNarrow>
__global__ __launch_bounds__(64 * W, 2) void gemm_i8_split_kernel(GemmI8Args g) {
    constexpr int kGroups = 64 / R;         // groups of 16 k in a step
    constexpr int kStep = 16 * kGroups;     // 32 or 64
    constexpr int kRegs = R * R / 64;       // result registers of an MFMA
    constexpr int kDepth = 3;               // steps in flight
    using acc_t = typename std::conditional<R == 32, v16i, v4i>::type;
    __shared__ __attribute__((aligned(16))) v4i part[W > 1 ? W : 1][W > 1 ? kRegs : 1][64];
    const int tile = tile_of_block(g);
    if (tile >= g.tiles || (int)(blockIdx.x >> 3) >= g.tiles_per_xcd) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane % R, group = lane / R;
    const int m0 = (tile % g.tiles_m) * R, n0 = (tile / g.tiles_m) * 4 * R;
    const char* a = g.a + (int64_t)blockIdx.z * g.a_batch;
    const char* b = g.b + (int64_t)blockIdx.z * g.b_batch;
    char* y = g.y + (int64_t)blockIdx.z * g.y_batch;

    const int n = n0 + 4 * col;  // the lane's four columns
    // (a dword at or past the end of a row: the row's last four bytes, shifted into place; columns past N are not stored)
    const int nb = n + 4 <= g.N ? n : g.N - 4;
    const int shift = n < g.N ? 8 * (n - nb) : 0;
    const bool ragged = !kNarrow && n0 + 4 * R > g.N;
    const uint32_t voff = (uint32_t)(group * 16) * (uint32_t)g.b_ld + (uint32_t)nb;
    const char* a_row = a + (int64_t)min(m0 + col, g.M - 1) * g.a_row;
    const char* b_col[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) b_col[i] = b + (int64_t)min(n + i, g.N - 1) * g.b_ld;

    const int32_t za = g.a_zp ? zero_point(g.a_zp, g.a_zp_signed) : g.a_zp_imm;
    const int32_t ca = (g.a_flip ? 128 : 0) - za;
    int32_t cb[4];
    bool any_cb = false;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        int32_t zb = g.b_zp_imm;
        if (g.b_zp) zb = zero_point(g.b_zp + (g.b_zp_len > 1 ? (int64_t)min(n + i, g.N - 1) * g.b_zp_stride : 0), g.b_zp_signed);
        cb[i] = (g.b_flip ? 128 : 0) - zb;
        any_cb = any_cb || cb[i] != 0;
    }
    any_cb = __builtin_amdgcn_ballot_w64(any_cb) != 0;

    acc_t acc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < kRegs; ++r) acc[i][r] = 0;
    int32_t col_sum[4] = {0, 0, 0, 0}, row_sum = 0;

    // what a step holds: the row of a, and b's dwords as loaded (or, b transposed, its fragments)
    struct Step {
        v4i fa;
        uint32_t w[16];
    };
    auto load = [&](auto tail_c, int step, Step& s) {
        constexpr bool kTail = decltype(tail_c)::value;
        const int k0 = step * kStep + group * 16;
        s.fa = load_k16<kTail>(a_row, k0, g.K);
        if constexpr (kBT) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const v4i v = load_k16<kTail>(b_col[i], k0, g.K);
#pragma unroll
                for (int e = 0; e < 4; ++e) s.w[4 * i + e] = (uint32_t)v[e];
            }
        } else {
            load_rows16<kTail, kNarrow>(b, b + (int64_t)(step * kStep) * g.b_ld, g.b_ld, voff, k0, g.K, g.N, s.w);
        }
    };
    auto multiply = [&](auto tail_c, int step, Step& s) {
        constexpr bool kTail = decltype(tail_c)::value;
        const int k0 = step * kStep + group * 16;
        const v4i fa = flipped<kTail>(s.fa, g.a_flip, k0, g.K);
        v4i fb[4];
        if constexpr (kBT) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                fb[i] = flipped<kTail>(v4i{(int)s.w[4 * i], (int)s.w[4 * i + 1], (int)s.w[4 * i + 2], (int)s.w[4 * i + 3]}, g.b_flip, k0, g.K);
        } else {
            columns_of<kTail>(s.w, ragged, shift, g.b_flip, k0, g.K, fb);
        }
        if (ca != 0) {
#pragma unroll
            for (int i = 0; i < 4; ++i) col_sum[i] = sum_bytes(fb[i], col_sum[i]);
        }
        if (any_cb) row_sum = sum_bytes(fa, row_sum);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (R == 32) acc[i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa, fb[i], acc[i], 0, 0, 0);
            else acc[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa, fb[i], acc[i], 0, 0, 0);
        }
    };

    const int full = g.K / kStep, steps = (g.K + kStep - 1) / kStep;
    const int per = (steps + W - 1) / W, lo = wave * per, hi = min(steps, lo + per), full_hi = min(full, hi);
    using no_tail = std::integral_constant<bool, false>;
    using tail = std::integral_constant<bool, true>;
    // The loads past this wavefront's last step read that step again: without a branch around them the compiler counts
    // the outstanding ones and waits for the oldest only.
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

    // the zero points' share of this wavefront's part of the sum
    auto over_groups = [&](int32_t v) {
        if (R == 16) v += __shfl_xor(v, 16);
        return v + __shfl_xor(v, 32);
    };
    if (ca != 0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int32_t add = ca * over_groups(col_sum[i]);
#pragma unroll
            for (int r = 0; r < kRegs; ++r) acc[i][r] += add;
        }
    }
    // lane: columns n .. n+3, rows row_of(r)
    auto row_of = [&](int r) { return (r / 4) * (4 * kGroups) + group * 4 + r % 4; };
    if (any_cb) {
        const int32_t mine = over_groups(row_sum) + (wave == 0 ? g.K * ca : 0);
#pragma unroll
        for (int r = 0; r < kRegs; ++r) {
            const int32_t of_row = __shfl(mine, row_of(r));
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i][r] += cb[i] * of_row;
        }
    }
    if constexpr (W == 1) {
        store_all<kRegs>(g, y, n, kRegs, [&](int r) { return m0 + row_of(r); }, [&](int r) { return v4i{acc[0][r], acc[1][r], acc[2][r], acc[3][r]}; });
    } else {
#pragma unroll
        for (int r = 0; r < kRegs; ++r) part[wave][r][lane] = v4i{acc[0][r], acc[1][r], acc[2][r], acc[3][r]};
        __syncthreads();
        constexpr int kMine = (kRegs + W - 1) / W;  // register r0 = wave, wave + W, ... of every wavefront's
        store_all<kMine>(g, y, n, kRegs >= W || wave < kRegs ? kMine : 0, [&](int i) { return m0 + row_of(i * W + wave); }, [&](int i) {
            const int r = i * W + wave;
            v4i sum = part[0][r][lane];
#pragma unroll
            for (int w = 1; w < W; ++w) sum += part[w][r][lane];
            return sum;
        });
    }
}

// Tile of 256 rows x 128 columns per work-group of four wavefronts, each with 64 rows.  K in steps of 128: every
// wavefront fetches and transposes the columns of one quarter of the step and leaves them in LDS, where all four read
// them (lane for lane as they were written: no bank conflicts); a's fragments have one reader each and come straight
// from memory.  Two steps in flight in registers, two LDS stages, one barrier per step.  For large products, where the
// wavefronts of the split kernel would transpose b once each: 4096 x 4096 x 4096 in 125 us (1100 TOP/s) against 176.
template <bool kBT>
__global__ __launch_bounds__(256) void gemm_i8_tile_kernel(GemmI8Args g) {
    constexpr int MT = 2;  // MFMA tiles along a wavefront's rows
    __shared__ __attribute__((aligned(16))) v4i sb[2][4][4][64];  // [stage][quarter of the step][column 4j + i][lane]
    const int tile = tile_of_block(g);
    if (tile >= g.tiles || (int)(blockIdx.x >> 3) >= g.tiles_per_xcd) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 31, group = lane >> 5;
    // Tiles go in bands of eight along M, n slowest inside: the 32 that an XCD has at a time read 8 runs of rows and 4 of
    // columns (with m alone fastest 32 runs of rows, more than its 4 MB of L2 from K = 512 on; 8192 x 1024 x 8192 184 -> 171 us)
    const int tiles_n = g.tiles / g.tiles_m, band = tile / (8 * tiles_n), in_band = tile - band * 8 * tiles_n, height = min(8, g.tiles_m - 8 * band);
    const int m0 = ((8 * band + in_band % height) * 4 + wave) * 32 * MT, n0 = (in_band / height) * 128;
    const char* a = g.a + (int64_t)blockIdx.z * g.a_batch;
    const char* b = g.b + (int64_t)blockIdx.z * g.b_batch;
    char* y = g.y + (int64_t)blockIdx.z * g.y_batch;
    const int n = n0 + 4 * col;
    const int nb = n + 4 <= g.N ? n : g.N - 4;
    const int shift = n < g.N ? 8 * (n - nb) : 0;
    const bool ragged = n0 + 128 > g.N;
    const uint32_t voff = (uint32_t)(group * 16) * (uint32_t)g.b_ld + (uint32_t)nb;
    const char* a_row[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) a_row[t] = a + (int64_t)min(m0 + 32 * t + col, g.M - 1) * g.a_row;
    const char* b_col[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) b_col[i] = b + (int64_t)min(n + i, g.N - 1) * g.b_ld;
    const int32_t za = g.a_zp ? zero_point(g.a_zp, g.a_zp_signed) : g.a_zp_imm;
    const int32_t ca = (g.a_flip ? 128 : 0) - za;
    const bool any_cb = g.b_zp_len > 1 || (g.b_flip ? 128 : 0) != (g.b_zp ? zero_point(g.b_zp, g.b_zp_signed) : g.b_zp_imm);

    struct Step {
        v4i a[MT][4];
        uint32_t w[16];
    };
    auto load = [&](auto tail_c, int step, Step& s) {
        constexpr bool kTail = decltype(tail_c)::value;
        const int k0 = step * 128 + group * 16;
        if constexpr (kBT) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const v4i v = load_k16<kTail>(b_col[i], k0 + wave * 32, g.K);
#pragma unroll
                for (int e = 0; e < 4; ++e) s.w[4 * i + e] = (uint32_t)v[e];
            }
        } else {
            load_rows16<kTail, false>(b, b + (int64_t)(step * 128 + wave * 32) * g.b_ld, g.b_ld, voff, k0 + wave * 32, g.K, g.N, s.w);
        }
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) s.a[t][e] = load_k16<kTail>(a_row[t], k0 + e * 32, g.K);
    };
    int32_t col_sum[4] = {0, 0, 0, 0}, row_sum[MT] = {};
    auto share = [&](auto tail_c, int step, int stage, Step& s) {
        constexpr bool kTail = decltype(tail_c)::value;
        const int k0 = step * 128 + group * 16 + wave * 32;
        v4i fb[4];
        if constexpr (kBT) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                fb[i] = flipped<kTail>(v4i{(int)s.w[4 * i], (int)s.w[4 * i + 1], (int)s.w[4 * i + 2], (int)s.w[4 * i + 3]}, g.b_flip, k0, g.K);
        } else {
            columns_of<kTail>(s.w, ragged, shift, g.b_flip, k0, g.K, fb);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) sb[stage][wave][i][lane] = fb[i];
        if (ca != 0) {
#pragma unroll
            for (int i = 0; i < 4; ++i) col_sum[i] = sum_bytes(fb[i], col_sum[i]);
        }
    };
    v16i acc[MT][4];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[t][i][r] = 0;
    auto multiply = [&](auto tail_c, int step, int stage, const Step& s) {
        constexpr bool kTail = decltype(tail_c)::value;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v4i fa[MT];
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                fa[t] = flipped<kTail>(s.a[t][e], g.a_flip, step * 128 + group * 16 + e * 32, g.K);
                if (any_cb) row_sum[t] = sum_bytes(fa[t], row_sum[t]);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const v4i fb = sb[stage][e][i][lane];
#pragma unroll
                for (int t = 0; t < MT; ++t) acc[t][i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[t], fb, acc[t][i], 0, 0, 0);
            }
        }
    };
    using no_tail = std::integral_constant<bool, false>;
    using tail = std::integral_constant<bool, true>;
    const int full = g.K / 128;
    if (full > 0) {
        // (the loads past the last step read it again, see the split kernel)
        Step s0, s1;
        load(no_tail(), 0, s0);
        load(no_tail(), min(1, full - 1), s1);
        int s = 0;
        for (; s + 2 <= full; s += 2) {
            share(no_tail(), 0, 0, s0);
            __syncthreads();
            multiply(no_tail(), 0, 0, s0);
            load(no_tail(), min(s + 2, full - 1), s0);
            share(no_tail(), 0, 1, s1);
            __syncthreads();
            multiply(no_tail(), 0, 1, s1);
            load(no_tail(), min(s + 3, full - 1), s1);
        }
        if (s < full) {
            share(no_tail(), 0, 0, s0);
            __syncthreads();
            multiply(no_tail(), 0, 0, s0);
        }
    }
    if (full * 128 < g.K) {
        Step last;
        load(tail(), full, last);
        share(tail(), full, full & 1, last);
        __syncthreads();
        multiply(tail(), full, full & 1, last);
    }

    int32_t cb[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        int32_t zb = g.b_zp_imm;
        if (g.b_zp) zb = zero_point(g.b_zp + (g.b_zp_len > 1 ? (int64_t)min(n + i, g.N - 1) * g.b_zp_stride : 0), g.b_zp_signed);
        cb[i] = (g.b_flip ? 128 : 0) - zb;
    }
    if (ca != 0) {
        // every wavefront has summed its quarters: the four sums of a column meet in LDS
        __syncthreads();
        int32_t* sums = reinterpret_cast<int32_t*>(&sb[0][0][0][0]);  // [4][128]
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int32_t both = col_sum[i] + __shfl_xor(col_sum[i], 32);
            if (group == 0) sums[wave * 128 + 4 * col + i] = both;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            int32_t add = 0;
            for (int w = 0; w < 4; ++w) add += sums[w * 128 + 4 * col + i];
            add *= ca;
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[t][i][r] += add;
        }
    }
    auto row_of = [&](int r) { return (r / 4) * 8 + group * 4 + r % 4; };
    if (any_cb) {
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            const int32_t mine = row_sum[t] + __shfl_xor(row_sum[t], 32) + g.K * ca;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int32_t of_row = __shfl(mine, row_of(r));
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[t][i][r] += cb[i] * of_row;
            }
        }
    }
    store_all<16 * MT>(g, y, n, 16 * MT, [&](int r) { return m0 + 32 * (r / 16) + row_of(r % 16); },
                       [&](int r) { return v4i{acc[r / 16][0][r % 16], acc[r / 16][1][r % 16], acc[r / 16][2][r % 16], acc[r / 16][3][r % 16]}; });
}

template <int R, int W>
void launch_split(const GemmI8Args& g, bool b_transposed, dim3 grid, hipStream_t s) {
    if (b_transposed) gemm_i8_split_kernel<R, W, true, false><<<grid, 64 * W, 0, s>>>(g);
    else if (g.N < 4) gemm_i8_split_kernel<R, W, false, true><<<grid, 64 * W, 0, s>>>(g);
    else gemm_i8_split_kernel<R, W, false, false><<<grid, 64 * W, 0, s>>>(g);
}

}  // namespace

int launch_matmul_i8(const MatMulDirectArgs& m, bool rne, hipStream_t s) {
    if (m.total == 0) return CHX_HIP_OK;
    const int64_t es = m.requant ? 1 : 4;
    const bool b_rows = m.b_col == 1 || m.N == 1, b_transposed = !b_rows && m.b_row == 1;
    // 16 bytes of every row are read at once; offsets within 16 rows of b are 32 bits wide; the sum of 2^31 products
    // is the direct kernel's (modulo 2^32) in any case
    if (m.K < 16 || m.a_col != 1 || !(b_rows || b_transposed) || (m.N > 1 && m.y_col != es)) return CHX_HIP_EUNSUPPORTED;
    if (m.a_zp_len > 1) return CHX_HIP_EUNSUPPORTED;  // a zero point per k
    const int64_t b_ld = b_rows ? m.b_row : m.b_col;
    if (m.M >= (int64_t(1) << 30) || m.N >= (int64_t(1) << 30) || m.K >= (int64_t(1) << 30) || b_ld < 0 || (b_rows && b_ld >= (int64_t(1) << 24))) return CHX_HIP_EUNSUPPORTED;
    if (b_rows && m.N < 4 && b_ld < m.N) return CHX_HIP_EUNSUPPORTED;  // rows that overlap: the narrow reads assume ascending ones
    const int64_t batch = m.total / (m.M * m.N);
    if (batch > 65535) return CHX_HIP_EUNSUPPORTED;
    GemmI8Args g;
    memset(&g, 0, sizeof(g));
    g.a = m.a; g.b = m.b; g.y = m.y;
    g.a_batch = m.a_batch; g.a_row = m.a_row; g.b_batch = m.b_batch; g.b_ld = b_ld; g.y_batch = m.y_batch; g.y_row = m.y_row;
    g.M = (int32_t)m.M; g.N = (int32_t)m.N; g.K = (int32_t)m.K;
    g.a_flip = m.a_signed ? 0u : 0x80808080u;
    g.b_flip = m.b_signed ? 0u : 0x80808080u;
    g.a_zp = m.a_zp_len ? m.a_zp : nullptr; g.a_zp_signed = m.a_zp_signed; g.a_zp_imm = m.a_zp_imm;
    g.b_zp = m.b_zp_len ? m.b_zp : nullptr; g.b_zp_len = m.b_zp_len; g.b_zp_stride = m.b_zp_stride; g.b_zp_signed = m.b_zp_signed; g.b_zp_imm = m.b_zp_imm;
    g.requant = m.requant; g.rne = rne ? 1 : 0; g.b_scale = m.b_scale; g.bias = m.bias; g.rq = m.rq;
    if (m.requant) {
        const QuantParams& q = m.rq.q;
        const double largest = 0x1p31 * fabs((double)m.rq.x_scale * (double)m.b_scale);  // of the values to be quantized
        g.finish = kExact;
        if (q.scale > 1e-20f && q.scale < 1e20f && largest < 1e30 && largest / (double)q.scale < 1e30) {
            g.inv_y_scale = 1.0f / q.scale;
            g.lo_folded = fold_relu_floor(q, m.rq.relu_floor, rne);
            g.qp = product_form(q, g.lo_folded, rne);
            g.finish = rne ? kFoldedRne : g.qp.path;
        }
    }
    auto tiles = [&](int tm, int tn) {
        g.tiles_m = (int32_t)((m.M + tm - 1) / tm);
        const int64_t t = (int64_t)g.tiles_m * ((m.N + tn - 1) / tn);
        g.tiles = (int32_t)t;
        g.tiles_per_xcd = (int32_t)((t + 7) / 8);
        return t;
    };
    if (((m.M + 15) / 16) * ((m.N + 63) / 64) >= (int64_t(1) << 28)) return CHX_HIP_EUNSUPPORTED;
    auto grid = [&]() { return dim3((unsigned)(8 * g.tiles_per_xcd), 1, (unsigned)batch); };
    // A compute unit for every tile, and K long enough that the loop, not the start and the result, is the time.  us on the
    // split kernel / on this one, int32 results and codes:
    //                        K = 256                     512                      768                       1024
    //    2048 x K x 4096   13.3 / 14.2  12.8 / 13.0   16.6 / 17.1  17.2 / 16.4   21.7 / 20.8  22.9 / 20.1   25.6 / 23.4  26.0 / 22.8
    //    4096 x K x 4096   20.9 / 27.4  19.3 / 22.5   29.7 / 34.0  30.3 / 29.6   40.9 / 40.6  40.7 / 36.7   49.1 / 45.7  47.8 / 41.8
    //    8192 x K x 8192   70.0 / 89.8  60.0 / 76.4    105 / 118    101 / 105     151 / 148    142 / 133     181 / 171    171 / 154
    //   16384 x K x 1024   22.0 / 27.3  20.2 / 22.0   32.2 / 33.7  30.7 / 28.7   45.1 / 41.3  41.1 / 36.0
    if (m.N >= 4 && m.K >= 768 && tiles(256, 128) * batch >= 256) {
        if (b_transposed) gemm_i8_tile_kernel<true><<<grid(), 256, 0, s>>>(g);
        else gemm_i8_tile_kernel<false><<<grid(), 256, 0, s>>>(g);
        return launch_check("gemm_i8_tile_kernel");
    }
    // Tiles of 16 x 64 where those of 32 x 128 would not give half the compute units work: 7.0 against 11.9 us for
    // 1 x 4096 x 4096 (floor 3.3: the bytes of b), 6.0 against 9.5 for 197 x 770 x 1001; with 256 tiles of 32 x 128
    // (1024 x 1024 x 1024) it is 8.3 against 7.2.
    const bool small = m.M <= 16 || tiles(32, 128) * batch <= 128;
    const int64_t work_groups = tiles(small ? 16 : 32, small ? 64 : 128) * batch, steps = (m.K + (small ? 63 : 31)) / (small ? 64 : 32);
    // K is split until every SIMD has two wavefronts (more only add to the sum at the end) or a wavefront one step
    int w = 1;
    while (w < 8 && 2 * w <= steps && 2 * w * work_groups <= 2048) w *= 2;
    if (small) {
        if (w == 1) launch_split<16, 1>(g, b_transposed, grid(), s);
        else if (w == 2) launch_split<16, 2>(g, b_transposed, grid(), s);
        else if (w == 4) launch_split<16, 4>(g, b_transposed, grid(), s);
        else launch_split<16, 8>(g, b_transposed, grid(), s);
    } else {
        if (w == 1) launch_split<32, 1>(g, b_transposed, grid(), s);
        else if (w == 2) launch_split<32, 2>(g, b_transposed, grid(), s);
        else if (w == 4) launch_split<32, 4>(g, b_transposed, grid(), s);
        else launch_split<32, 8>(g, b_transposed, grid(), s);
    }
    return launch_check("gemm_i8_split_kernel");
}

}  // namespace chx
