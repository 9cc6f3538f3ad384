// Integer matrix products on the int8 matrix cores: MatMulInteger and QLinearMatMul.
//
//   y[m, n] = sum_k (a[m, k] - za) * (b[k, n] - zb[n])      exact int32; then the int32 itself, or the requantized code
//
// Both operands are read as they are: nothing is packed, expanded or copied first, no scratch memory, no value that
// the host has to read back (the zero points are fetched by the kernel), so a call is one launch, also inside a
// recorded run.
//
// Fragments of the split kernel (the staged one has them from LDS).  v_mfma_i32_32x32x32_i8 wants 16 consecutive k of one row (column) per lane.  A row of a has them in
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
#include <algorithm>
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
    uint32_t turn;  // 1: some XCD would have no tile (tile_of_block)
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

// The (ONNX) bias of four neighbouring columns: added to the sum.
__device__ __forceinline__ v4i bias4(const GemmI8Args& g, int n) {
    v4i bias = {0, 0, 0, 0};
    if (g.bias) {
#pragma unroll
        for (int i = 0; i < 4; ++i) bias[i] = g.bias[n + i < g.N ? n + i : g.N - 1];
    }
    return bias;
}

// A lane's results in kCount rows: sum(i) gives the four of row(i), for i < count (the same in every lane); bias() is asked for codes only.
template <int kCount, class Row, class Sum, class Bias>
__device__ __forceinline__ void store_all(const GemmI8Args& g, char* y, int n, int count, Row row, Sum sum, Bias bias_of) {
    if (!g.requant) {
#pragma unroll
        for (int i = 0; i < kCount; ++i)
            if (i < count) store4(g, y, row(i), n, sum(i));
        return;
    }
    const v4i bias = bias_of();
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
// that read the same columns of b find them in one L2.  Where that leaves XCDs
// without a tile, the runs move on by one XCD from product to product of a batch (851 products of one tile 29 us and 17 this way;
// 43 of ten tiles 8.8 and 8.3; 19 of 24 tiles, which leave none, 5.5 and 6.0).
__device__ __forceinline__ int tile_of_block(const GemmI8Args& g) {
    return (int)((blockIdx.x + blockIdx.z * g.turn) & 7) * g.tiles_per_xcd + (int)(blockIdx.x >> 3);
}

// Tile of R rows x 4R columns per work-group (R = 16 or 32); its W wavefronts share K out and add their sums through LDS at the end.
// No LDS on the way in: a wavefront's fragments come straight from memory, three K steps ahead in registers.  Bound by
// latency (a step costs about a microsecond when nothing hides it, so K is split and the loads run ahead) and, with many
// tiles, by the vector instructions of the transposition.  One thread per result, K serial, took 160 us for
// 197 x 770 x 1001; this 5.6.
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
        store_all<kRegs>(g, y, n, kRegs, [&](int r) { return m0 + row_of(r); }, [&](int r) { return v4i{acc[0][r], acc[1][r], acc[2][r], acc[3][r]}; },
                         [&]() { return bias4(g, n); });
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
        }, [&]() { return bias4(g, n); });
    }
}

typedef int v2i __attribute__((ext_vector_type(2)));

// Eight rows of sixteen bytes in LDS, transposed: in a group of 16 lanes, lanes 2r and 2r + 1 give the two halves of row r, lane j gets column j.
__device__ __forceinline__ v2i transposed8(const char* p) {
    typedef __attribute__((address_space(3))) v2i* Lds;
    return __builtin_amdgcn_ds_read_tr8_b64_v2i32((Lds)(uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)p);
}

// Tile of 64 kRW rows x 64 kCW columns per work-group of eight wavefronts; kKW of them share out the K of a stage (128, or 256
// with eight).  Every thread brings 16 bytes of a row of a and 16 of a row of b at a time, coalesced and once per work-group,
// into one of two stages in LDS, one barrier per stage.  A fragment of a is a 16-byte read (rows an odd number of 16
// bytes apart; 0.1 to 0.4 conflict cycles per LDS instruction in all); one of b, whose rows run along n, comes out of ds_read_b64_tr_b8 transposed, without a vector
// instruction (b transposed: like a).  b is the first operand of the MFMA, so that a lane ends with four
// neighbouring results of a row.
//
// For products whose time is the loop: the split kernel transposes b once for every 32 rows, 48 vector instructions for four
// MFMAs, and reads unaligned rows in dwords.  Bound by LDS (96 KB of traffic for 128 x 128 x 128, 1.9 POP/s with a
// work-group per compute unit), and below about 10 stages by the start and the results.  us on the split kernel (the last three: on a tile kernel
// with the transposition in registers, deleted for this) and on this one, int32 results: 1024 x 1024 x 4096 16.3 and 13.0, with
// 4095 columns 22.8 and 14.1, 512 x 4096 x 1024 15.9 and 13.4, 128 x 4096 x 4096 17.5 and 13.2;
// 2048 x 1024 x 4096 22.0 and 17.0, 4096 x 4096 x 4096 118 and 90, 8192 x 1024 x 8192 156 and 116.
// At 128 registers two work-groups fit a compute unit: one's loop runs beside the other's start and end (4096 x 1024 x 4096: 38.9
// with two stages held in registers and 165 of them).
template <bool kBT, int kRW, int kCW, int kKW>
struct StageShape {
    static constexpr int kThreads = 64 * kRW * kCW * kKW, kRows = 64 * kRW, kCols = 64 * kCW;
    static constexpr int kK = kKW == 8 ? 256 : 128, kSub = kK / 32 / kKW;  // K of a stage; MFMA steps of a wavefront in it
    static constexpr int kAPitch = kK + 16, kBPitch = kBT ? kK + 16 : kCols == 64 ? 80 : kCols + 32;
    static constexpr int kABytes = kRows * kAPitch, kBBytes = kBT ? kCols * kBPitch : kK * kBPitch, kStage = kABytes + kBBytes;
    static constexpr int kAChunks = kRows * kK / 16 / kThreads, kBChunks = kCols * kK / 16 / kThreads;
    static constexpr int kParts = kThreads / 64 * 32 * 272;  // [wavefront][32 rows][64 columns, and 4 to keep off the banks] int32
    static constexpr int kLds = 2 * kStage > kParts + (kKW + 1) * (kRows + kCols) * 4 ? 2 * kStage : kParts + (kKW + 1) * (kRows + kCols) * 4;
};

// kShort: rows of b of 4 to 15 bytes (b not transposed).  The 16 bytes that are read of a row reach into the rows behind it, whose share of the result is
// stored nowhere; the last rows are read as the last 16 bytes of b and shifted.
template <bool kBT, int kRW, int kCW, int kKW, bool kShort>
__device__ __forceinline__ void stage_product(const GemmI8Args& g) {
    using S = StageShape<kBT, kRW, kCW, kKW>;
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int tile = tile_of_block(g);
    if (tile >= g.tiles || (int)(blockIdx.x >> 3) >= g.tiles_per_xcd) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, group = lane >> 5;
    const int rw = wave % kRW, cw = wave / kRW % kCW, kw = wave / (kRW * kCW);
    // Tiles go in bands of eight along M, n slowest inside: the 32 that an XCD has at a time read 8 runs of rows and 4 of
    // columns (with m alone fastest 32 runs of rows, more than its 4 MB of L2)
    const int tiles_n = g.tiles / g.tiles_m, band = tile / (8 * tiles_n), in_band = tile - band * 8 * tiles_n, height = min(8, g.tiles_m - 8 * band);
    const int m0 = (8 * band + in_band % height) * S::kRows, n0 = (in_band / height) * S::kCols;
    const char* a = g.a + (int64_t)blockIdx.z * g.a_batch;
    const char* b = g.b + (int64_t)blockIdx.z * g.b_batch;
    char* y = g.y + (int64_t)blockIdx.z * g.y_batch;

    // what this thread brings: 16 bytes of a row of a; of b 16 columns of one k (or, transposed, like a)
    constexpr int kAPerRow = S::kK / 16, kBPerRow = kBT ? S::kK / 16 : S::kCols / 16;
    const char* const a_tile = a + (int64_t)m0 * g.a_row;
    const char* const b_tile = kBT ? b + (int64_t)n0 * g.b_ld : b;
    uint32_t a_off[S::kAChunks], b_off[S::kBChunks];  // (the launcher has seen that they fit)
#pragma unroll
    for (int c = 0; c < S::kAChunks; ++c) a_off[c] = (uint32_t)min((tid + c * S::kThreads) / kAPerRow, g.M - 1 - m0) * (uint32_t)g.a_row + tid % kAPerRow * 16;
    const int b_n = n0 + tid % kBPerRow * 16, b_from = kShort ? 0 : min(b_n, g.N - 16);
    // the bytes by which a chunk that reaches past the end of its row is read too early (16 and more: it is past the end whole)
    const int b_shift = kBT ? 0 : b_n - b_from;
#pragma unroll
    for (int c = 0; c < S::kBChunks; ++c) {
        const int i = (tid + c * S::kThreads) / kBPerRow;
        b_off[c] = kBT ? (uint32_t)min(i, g.N - 1 - n0) * (uint32_t)g.b_ld + tid % kBPerRow * 16 : (uint32_t)i * (uint32_t)g.b_ld + b_from;
    }
    const bool ragged = !kBT && !kShort && n0 + S::kCols > g.N;
    // the bytes by which the 16 of row k would pass the end of b
    const int64_t b_bytes = (int64_t)(g.K - 1) * g.b_ld + g.N;
    auto past_b = [&](int k) { return (int)max(min(k, g.K - 1) * g.b_ld + 16 - b_bytes, (int64_t)0); };
    const int a_k = tid % kAPerRow * 16, b_k = kBT ? tid % kBPerRow * 16 : tid / kBPerRow;

    struct Stage {
        v4i a[S::kAChunks], b[S::kBChunks];
    };
    auto load = [&](auto tail_c, int stage, Stage& s) {
        constexpr bool kTail = decltype(tail_c)::value;
        const int k0 = stage * S::kK;
        const char* const from_a = a_tile + k0;
        const char* const from_b = b_tile + (kBT ? (int64_t)k0 : k0 * g.b_ld);
        // (the last stage: 16 bytes of a row that reach past K are its last 16, see load_k16; a row of b from K on is the last one)
#pragma unroll
        for (int c = 0; c < S::kBChunks; ++c) {
            const int k = k0 + b_k + (kBT ? 0 : c * (S::kThreads / kBPerRow));
            const char* p = from_b + b_off[c];
            if (kTail && kBT && k + 16 > g.K) p -= k + 16 - g.K;
            if (kTail && !kBT && k >= g.K) p -= (k + 1 - g.K) * g.b_ld;
            if (kShort) p -= past_b(k);
            s.b[c] = *reinterpret_cast<const v4i_u*>(p);
        }
#pragma unroll
        for (int c = 0; c < S::kAChunks; ++c) {
            const char* p = from_a + a_off[c];
            if (kTail && k0 + a_k + 16 > g.K) p -= k0 + a_k + 16 - g.K;
            s.a[c] = *reinterpret_cast<const v4i_u*>(p);
        }
    };
    auto share = [&](auto tail_c, int stage, int where, Stage& s) {
        constexpr bool kTail = decltype(tail_c)::value;
        const int k0 = stage * S::kK;
        char* const sa = lds + where * S::kStage;
        char* const sb = sa + S::kABytes;
#pragma unroll
        for (int c = 0; c < S::kBChunks; ++c) {
            const int i = tid + c * S::kThreads;
            v4i v = s.b[c];
            if constexpr (kBT) {
                v = flipped<kTail>(v, g.b_flip, k0 + b_k, g.K);
                *reinterpret_cast<v4i*>(sb + i / kBPerRow * S::kBPitch + b_k) = v;
            } else {
                if (ragged && b_shift > 0 && b_shift < 16) v = shift_down(v, b_shift);
                if (kShort) {
                    const int past = past_b(k0 + i / kBPerRow);
                    if (past > 0) v = shift_down(v, past);
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = kTail && k0 + i / kBPerRow >= g.K ? 0 : v[e] ^ (int)g.b_flip;
                *reinterpret_cast<v4i*>(sb + i / kBPerRow * S::kBPitch + i % kBPerRow * 16) = v;
            }
        }
#pragma unroll
        for (int c = 0; c < S::kAChunks; ++c)
            *reinterpret_cast<v4i*>(sa + (tid + c * S::kThreads) / kAPerRow * S::kAPitch + a_k) = flipped<kTail>(s.a[c], g.a_flip, k0 + a_k, g.K);
    };

    const int32_t za = g.a_zp ? zero_point(g.a_zp, g.a_zp_signed) : g.a_zp_imm;
    const int32_t ca = (g.a_flip ? 128 : 0) - za;
    const bool any_cb = g.b_zp_len > 1 || (g.b_flip ? 128 : 0) != (g.b_zp ? zero_point(g.b_zp, g.b_zp_signed) : g.b_zp_imm);
    // the four columns of which the lane stores results in the end, and what is fetched for them: with the last stage, so that it
    // is there in time and takes no registers before
    const int c = cw * 64 + lane % 16 * 4;
    v4i bias;
    int32_t cb[4];
    auto load_columns = [&]() {
        bias = g.requant ? bias4(g, n0 + c) : v4i{0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            int32_t zb = g.b_zp_imm;
            if (g.b_zp) zb = zero_point(g.b_zp + (g.b_zp_len > 1 ? (int64_t)min(n0 + c + i, g.N - 1) * g.b_zp_stride : 0), g.b_zp_signed);
            cb[i] = (g.b_flip ? 128 : 0) - zb;
        }
    };
    v16i acc[2][2];  // [columns][rows]
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i / 2][i % 2][r] = 0;
    int32_t col_sum[2] = {0, 0}, row_sum[2] = {0, 0};
    const int a_at = (rw * 64 + col) * S::kAPitch + kw * S::kSub * 32 + group * 16;
    const int b_at = S::kABytes + (kBT ? (cw * 64 + col) * S::kBPitch + kw * S::kSub * 32 + group * 16
                                       : (kw * S::kSub * 32 + group * 16 + (lane & 15) / 2) * S::kBPitch + cw * 64 + (lane >> 4 & 1) * 16 + (lane & 1) * 8);
    auto multiply = [&](int where) {
        const char* const base = lds + where * S::kStage;
#pragma unroll
        for (int sub = 0; sub < S::kSub; ++sub) {
            v4i fa[2], fb[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) fa[t] = *reinterpret_cast<const v4i*>(base + a_at + t * 32 * S::kAPitch + sub * 32);
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                if constexpr (kBT) {
                    fb[i] = *reinterpret_cast<const v4i*>(base + b_at + i * 32 * S::kBPitch + sub * 32);
                } else {
                    const v2i lo = transposed8(base + b_at + i * 32 + sub * 32 * S::kBPitch), hi = transposed8(base + b_at + i * 32 + (sub * 32 + 8) * S::kBPitch);
                    fb[i] = v4i{lo[0], lo[1], hi[0], hi[1]};
                }
            }
            if (ca != 0 && rw == 0) {
#pragma unroll
                for (int i = 0; i < 2; ++i) col_sum[i] = sum_bytes(fb[i], col_sum[i]);
            }
            if (any_cb && cw == 0) {
#pragma unroll
                for (int t = 0; t < 2; ++t) row_sum[t] = sum_bytes(fa[t], row_sum[t]);
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int t = 0; t < 2; ++t) acc[i][t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fb[i], fa[t], acc[i][t], 0, 0, 0);
        }
    };
    using no_tail = std::integral_constant<bool, false>;
    using tail = std::integral_constant<bool, true>;
    const int full = g.K / S::kK;
    const bool rest = full * S::kK < g.K;
    Stage held;
    if (full > 0) {
        load(no_tail(), 0, held);
        for (int s = 0; s + 1 < full; ++s) {
            share(no_tail(), s, s & 1, held);
            load(no_tail(), s + 1, held);
            __syncthreads();
            multiply(s & 1);
        }
        share(no_tail(), full - 1, (full - 1) & 1, held);
        if (rest) load(tail(), full, held);
        else load_columns();
        __syncthreads();
        multiply((full - 1) & 1);
    } else {
        load(tail(), 0, held);
    }
    if (rest) {
        share(tail(), full, full & 1, held);
        load_columns();
        __syncthreads();
        multiply(full & 1);
    }

    // ---- the zero points' share: the sums of the columns (rows) from the wavefronts that had them first ----
    int32_t* const sums = reinterpret_cast<int32_t*>(lds + S::kParts);  // [kKW][columns, rows], then the totals
    constexpr int kSums = S::kCols + S::kRows;
    __syncthreads();  // (the stages are read)
    if (ca != 0 || any_cb) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int32_t of_col = col_sum[i] + __shfl_xor(col_sum[i], 32), of_row = row_sum[i] + __shfl_xor(row_sum[i], 32);
            if (group == 0 && rw == 0) sums[kw * kSums + cw * 64 + i * 32 + col] = of_col;
            if (group == 0 && cw == 0) sums[kw * kSums + S::kCols + rw * 64 + i * 32 + col] = of_row;
        }
        __syncthreads();
        if (tid < kSums) {
            int32_t total = 0;
#pragma unroll
            for (int w = 0; w < kKW; ++w) total += sums[w * kSums + tid];
            sums[kKW * kSums + tid] = total;
        }
        __syncthreads();
    }
    const int32_t* const total = sums + kKW * kSums;
    v4i col_add = {0, 0, 0, 0};
    if (ca != 0) {
#pragma unroll
        for (int e = 0; e < 4; ++e) col_add[e] = ca * total[c + e];
    }
    // The sums of a tile's kKW wavefronts meet in LDS, 32 rows at a time, and leave it with 16 lanes along a row: 256 bytes of
    // results (64 of codes) in one place.  Straight from the registers, a lane has four results of each of many rows, and
    // the parts of lines cost more than everything else (4096 x 256 x 4096: 78 us against 20).
    // (twice, and not a loop: the compiler leaves one that long as it is, and the sums go to memory)
    auto finish = [&](auto which) {
        constexpr int t = decltype(which)::value, kMine = 8 / kKW;
        char* const mine = lds + wave * (32 * 272);
        if (t > 0 && kKW > 1) __syncthreads();
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const v16i& v = acc[u / 4][t];
            const int q = u % 4;
            *reinterpret_cast<v4i*>(mine + col * 272 + (u / 4 * 32 + q * 8 + group * 4) * 4) = v4i{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
        }
        if (kKW > 1) __syncthreads();
        const char* const parts = lds + (rw + kRW * cw) * (32 * 272);  // of the wavefronts kRW * kCW apart that share a tile
        auto row = [&](int j) { return (kw * kMine + j) * 4 + lane / 16; };
        store_all<kMine>(g, y, n0 + c, kMine, [&](int j) { return m0 + rw * 64 + t * 32 + row(j); }, [&](int j) {
            v4i sum = *reinterpret_cast<const v4i*>(parts + row(j) * 272 + lane % 16 * 16);
#pragma unroll
            for (int w = 1; w < kKW; ++w) sum += *reinterpret_cast<const v4i*>(parts + w * kRW * kCW * (32 * 272) + row(j) * 272 + lane % 16 * 16);
            sum += col_add;
            if (any_cb) {
                const int32_t of_row = total[S::kCols + rw * 64 + t * 32 + row(j)] + g.K * ca;
#pragma unroll
                for (int e = 0; e < 4; ++e) sum[e] += cb[e] * of_row;
            }
            return sum;
        }, [&]() { return bias; });
    };
    finish(std::integral_constant<int, 0>());
    finish(std::integral_constant<int, 1>());
}

// (launch bounds: 128 registers)
template <bool kBT, int kRW, int kCW, int kKW>
__global__ __launch_bounds__(64 * kRW * kCW * kKW, 4) void gemm_i8_stage_kernel(GemmI8Args g) {
    stage_product<kBT, kRW, kCW, kKW, false>(g);
}

template <int kRW, int kCW, int kKW>
__global__ __launch_bounds__(64 * kRW * kCW * kKW, 4) void gemm_i8_stage_short_kernel(GemmI8Args g) {
    stage_product<false, kRW, kCW, kKW, true>(g);
}

template <bool kBT, int kRW, int kCW, int kKW>
int launch_stage(const GemmI8Args& g, dim3 grid, hipStream_t s) {
    using S = StageShape<kBT, kRW, kCW, kKW>;
    if (S::kLds > 64 * 1024)  // (has to be asked for, on every device)
        CHX_HIP_CALL(hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_i8_stage_kernel<kBT, kRW, kCW, kKW>), hipFuncAttributeMaxDynamicSharedMemorySize, S::kLds));
    gemm_i8_stage_kernel<kBT, kRW, kCW, kKW><<<grid, S::kThreads, S::kLds, s>>>(g);
    return launch_check("gemm_i8_stage_kernel");
}

template <int kRW, int kCW, int kKW>
int launch_stage_short(const GemmI8Args& g, dim3 grid, hipStream_t s) {
    using S = StageShape<false, kRW, kCW, kKW>;
    CHX_HIP_CALL(hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_i8_stage_short_kernel<kRW, kCW, kKW>), hipFuncAttributeMaxDynamicSharedMemorySize, S::kLds));
    gemm_i8_stage_short_kernel<kRW, kCW, kKW><<<grid, S::kThreads, S::kLds, s>>>(g);
    return launch_check("gemm_i8_stage_short_kernel");
}

template <int R, int W>
void launch_split(const GemmI8Args& g, bool b_transposed, dim3 grid, hipStream_t s) {
    if (b_transposed) gemm_i8_split_kernel<R, W, true, false><<<grid, 64 * W, 0, s>>>(g);
    else if (g.N < 4) gemm_i8_split_kernel<R, W, false, true><<<grid, 64 * W, 0, s>>>(g);
    else gemm_i8_split_kernel<R, W, false, false><<<grid, 64 * W, 0, s>>>(g);
}

// Times in us, fitted to 14,000 products of 48 to 4096 rows, columns and K, int32 results and codes (within 4 % for the stage
// kernel, 10 % for the split kernel).  The choice they give makes those products 1.07 times as fast on average as the split
// kernel, 1.33 times with b transposed, and is within 1 % (3 %) of the best choice on average.
struct StageCost {
    double launch, stage, round, a_odd, second, b_odd, more;
};
struct SplitCost {
    double launch, step, a_odd, b_odd, filled, tail, results;
};
constexpr StageCost kStageCosts[2][3] = {
        {{5.5, 0.575, 1.80, 0.17, 1.18, 0.275, 1.9}, {3.25, 0.388, 2.74, 0.125, 0.765, 0.295, 1.51}, {4.1, 0.513, 2.13, 0.206, 0.977, 0.363, 1.47}},
        {{5.45, 0.520, 1.57, 0.39, 1.24, 0.04, 1.95}, {3.4, 0.352, 2.73, 0.48, 0.82, 0.03, 1.49}, {3.57, 0.371, 2.34, 0.84, 0.83, 0.05, 1.47}}};
constexpr SplitCost kSplitCosts[2] = {{4.32, 0.56, 0.375, 0.405, 0.134, 0.09, 0.39}, {3.76, 1.00, 1.13, 0.02, 0.142, 0.0, 0.44}};

// `tiles` of the work-groups' size, `stages` of K; odd: rows that are no whole dwords; two work-groups share a compute unit
double stage_time(const StageCost& c, double tiles, double stages, bool a_odd, bool b_odd) {
    const double rounds = tiles <= 256 ? 1.0 : (1.0 + c.second) * (tiles <= 512 ? 1.0 : std::max(tiles / 512.0, c.more));
    return c.launch + rounds * (stages * c.stage * (a_odd ? 1.0 + c.a_odd : 1.0) * (b_odd ? 1.0 + c.b_odd : 1.0) + c.round);
}

// `steps` of a wavefront, `filled`: wavefronts per SIMD
double split_time(const SplitCost& c, double steps, double filled, bool a_odd, bool b_odd, bool tail, double results) {
    return c.launch + steps * (c.step + c.filled * filled) * (a_odd ? 1.0 + c.a_odd : 1.0) * (b_odd ? 1.0 + c.b_odd : 1.0) + (tail ? c.tail : 0.0) + results * 1e-6 * c.results +
           (results > 16e6 ? (results - 16e6) * 0.6e-6 : 0.0);  // (more than the caches hold: 8192 x 512 x 8192 101 us)
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
        g.turn = (int64_t)g.tiles_per_xcd * 7 >= t ? 1 : 0;
        return t;
    };
    if (((m.M + 15) / 16) * ((m.N + 63) / 64) >= (int64_t(1) << 28)) return CHX_HIP_EUNSUPPORTED;
    auto grid = [&]() { return dim3((unsigned)(8 * g.tiles_per_xcd), 1, (unsigned)batch); };
    // Tiles of 16 x 64 where those of 32 x 128 would not give half the compute units work: 7.0 against 11.9 us for
    // 1 x 4096 x 4096 (floor 3.3: the bytes of b), 6.0 against 9.5 for 197 x 770 x 1001; with 256 tiles of 32 x 128
    // (1024 x 1024 x 1024) it is 8.3 against 7.2.
    const bool small = m.M <= 16 || tiles(32, 128) * batch <= 128;
    const int64_t work_groups = tiles(small ? 16 : 32, small ? 64 : 128) * batch, steps = (m.K + (small ? 63 : 31)) / (small ? 64 : 32);
    // K is split until every SIMD has two wavefronts (more only add to the sum at the end) or a wavefront one step
    int w = 1;
    while (w < 8 && 2 * w <= steps && 2 * w * work_groups <= 2048) w *= 2;
    // The stage kernel with tiles of 128 x 128, 64 x 128 or 64 x 64 where its time is the shortest by the fits above and a tenth below
    // the split kernel's, whose fit is the coarser one (then one product in 200 gets slower by more than 3 %, and with less
    // than three steps for a wavefront, which the split kernel has in flight at once, none).  A row's 16 bytes are read in one
    // place, offsets in a tile are 32 bits wide, and one stage is no loop.  (Below 2^26 products the start is the time on either.)
    // The fits end at 4096 rows and take codes and int32 for one.  With b as it lies, K of 192 (to codes also 256 and 320) and rows of y in
    // whole lines that counts: two or three stages are no pipeline, and the split kernel's results leave sooner, codes most of all.  Split and
    // stage in us: 8192 x 192 x 4096 to codes 29.4 and 33.9, 18612 x 192 x 2944 51 and 58, 32768 x 256 x 4096 112 and 117; to int32 100352 x 192 x 256 28.6 and
    // 31.8, but 65180 x 256 x 128 13.6 and 11.6; from K 352 on stage is faster (8192 x 384 x 1024 6 % and 12 %).  The fits hold where the split
    // kernel has a rest of K (26288 x 252 x 2944 to codes 85 and 75) and for rows that do not begin lines, of which its tiles write parts
    // (49490 x 240 x 2712 152 and 129).
    const bool short_k = !b_transposed && m.K % 64 == 0 && m.K <= (m.requant ? 320 : 192) && m.y_row % 128 == 0;
    const int64_t steps_each = (steps + w - 1) / w;
    if (!m.lds_64k && !short_k && steps_each > 2 && m.N >= 16 && m.K >= 192 && (double)(m.M * m.N) * (double)(m.K * batch) >= 0x1p26 && m.a_row >= 0 && m.a_row < (int64_t(1) << 24) && b_ld < (int64_t(1) << 24)) {
        const bool a_odd = m.K % 4 != 0, b_odd = m.N % 4 != 0;
        const int64_t along_m[3] = {128, 64, 64}, along_n[3] = {128, 128, 64};
        // (the split kernel's fit does not know operands that leave the caches: 27015 x 4416 x 3968 to codes 555 us by it, 1,160 in truth)
        const bool filled = m.K >= 768 && ((m.M + 255) / 256) * ((m.N + 127) / 128) * batch >= 256;
        double least = filled ? 1e30 : 0.9 * split_time(kSplitCosts[b_transposed], (double)steps_each, (double)(work_groups * w) / 1024.0, a_odd, b_odd,
                                         m.K % (small ? 64 : 32) != 0, (double)m.M * (double)m.N * (double)batch);
        int best = -1;
        for (int i = 0; i < 3; ++i) {
            const double t = stage_time(kStageCosts[b_transposed][i], (double)(tiles((int)along_m[i], (int)along_n[i]) * batch), (double)((m.K + (i == 2 ? 255 : 127)) / (i == 2 ? 256 : 128)), a_odd, b_odd);
            if (t < least) {
                least = t;
                best = i;
            }
        }
        // (the fits are of single products.  In batches with a K of two or three stages, a round or two of tiles that are mostly padding have little beside their start: 17 x 638 x 295 x 146
        // 10.3 us split and 13.7, 454 x 68 x 259 x 21 32 and 41; of 37 drawn batches of such K nine were slower by more than 3 %, seven of them these;
        // of 289 others by this choice nine, by up to 22 %, and 0.71 of the time on average)
        if (best == 0 && batch > 1 && !b_transposed && m.K < 400 && tiles(128, 128) * batch <= 512 && 1.6 * (double)(m.M * m.N) < 16384.0 * (double)g.tiles) best = -1;
        if (best >= 0) {
            (void)tiles((int)along_m[best], (int)along_n[best]);
            if (best == 0) return b_transposed ? launch_stage<true, 2, 2, 2>(g, grid(), s) : launch_stage<false, 2, 2, 2>(g, grid(), s);
            if (best == 1) return b_transposed ? launch_stage<true, 1, 2, 4>(g, grid(), s) : launch_stage<false, 1, 2, 4>(g, grid(), s);
            return b_transposed ? launch_stage<true, 1, 1, 8>(g, grid(), s) : launch_stage<false, 1, 1, 8>(g, grid(), s);
        }
        (void)tiles(small ? 16 : 32, small ? 64 : 128);
    }
    // Fewer than 16 columns, which the choice above leaves out, and a compute unit for every 256 rows: the split kernel reads (and transposes) b for every 32
    // rows of a.  us there and in tiles of 128 x 64: 110767 x 3583 x 15 404 and 117, 181346 x 907 x 15 129 and 44, 304796 x 2322 x 6 to codes 517 and 166; with b transposed
    // 229322 x 1723 x 8 to codes 310 and 105, 359525 x 2641 x 4 739 and 253.
    if (!m.lds_64k && m.N >= 4 && m.N < 16 && m.K >= 768 && ((m.M + 255) / 256) * batch >= 256 && m.a_row >= 0 && m.a_row < (int64_t(1) << 24) && (b_transposed ? b_ld < (int64_t(1) << 24) : b_ld >= m.N)) {
        (void)tiles(128, 64);
        return b_transposed ? launch_stage<true, 2, 1, 4>(g, grid(), s) : launch_stage_short<2, 1, 4>(g, grid(), s);
    }
    // (few products of one tile start sooner on one XCD, which has two wavefronts per SIMD for 256: 63 x 4 x 100 x 11 3.7 us and 4.2 on all, 219 x
    // 10 x 23 x 11 4.6 and 4.9, 258 wavefronts of 129 x 29 x 83 x 45 0.7 of the time on all)
    if (g.tiles == 1 && batch * w <= 256) g.turn = 0;
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
