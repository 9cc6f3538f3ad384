// Device-side pieces of the integer products that read their operands as they lie in memory (gemm_i8.hip,
// conv_planar.hip).  Internal linkage: each translation unit gets its own copy.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace chx {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
// the same with no alignment: one global_load_dwordx4 / global_load_dword each (unaligned access is on for this target)
typedef int v4i_u __attribute__((ext_vector_type(4), aligned(1)));
typedef uint32_t u32_u __attribute__((aligned(1)));

__device__ __forceinline__ int32_t zero_point(const char* p, int32_t is_signed) {
    const uint8_t raw = *reinterpret_cast<const uint8_t*>(p);
    return is_signed ? (int32_t)(int8_t)raw : (int32_t)raw;
}

// v >> (8 * bytes), zeros moving in; 1 <= bytes <= 15
__device__ __forceinline__ v4i shift_down(v4i v, int bytes) {
    uint64_t lo = (uint32_t)v[0] | (uint64_t)(uint32_t)v[1] << 32, hi = (uint32_t)v[2] | (uint64_t)(uint32_t)v[3] << 32;
    const int s = 8 * bytes;
    if (s >= 64) {
        lo = hi >> (s - 64);
        hi = 0;
    } else {
        lo = lo >> s | hi << (64 - s);
        hi >>= s;
    }
    return v4i{(int)(uint32_t)lo, (int)(lo >> 32), (int)(uint32_t)hi, (int)(hi >> 32)};
}

// 16 consecutive k of one row, as they lie in memory; kTail: k0 may be near or past K (what is read then is not the
// row's, and fix_tail puts it right)
template <bool kTail>
__device__ __forceinline__ v4i load_k16(const char* row, int k0, int K) {
    return *reinterpret_cast<const v4i_u*>(row + (kTail && k0 + 16 > K ? K - 16 : k0));
}

// sign bits flipped, and for a group at the end of K: the bytes from K on zero
template <bool kTail>
__device__ __forceinline__ v4i flipped(v4i v, uint32_t flip, int k0, int K) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] ^= (int)flip;
    if (!kTail || k0 + 16 <= K) return v;
    return k0 < K ? shift_down(v, 16 - (K - k0)) : v4i{0, 0, 0, 0};
}

// 16 rows of a lane's four columns, as they lie in memory: row i of them is k0 + i (kTail: 0 for rows from K on).
// `at`, the same in every lane, is where the step's first row starts; `voff` the lane's offset from there (its own group
// of rows, its columns): the addresses then cost scalar instructions only.
// kNarrow: fewer than four columns; a dword reaches into the following rows, and the last ones are read as the last
// four bytes of b and shifted.
template <bool kTail, bool kNarrow>
__device__ __forceinline__ void load_rows16(const char* b, const char* at, int64_t ld, uint32_t voff, int k0, int K, int N, uint32_t (&w)[16]) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        if (kTail) {
            w[i] = 0;
            if (k0 + i >= K) continue;
        }
        if (kNarrow) {
            const int64_t row = (int64_t)(k0 + i) * ld, last = (int64_t)(K - 1) * ld + N - 4;
            w[i] = *reinterpret_cast<const u32_u*>(b + (row < last ? row : last)) >> (row < last ? 0 : 8 * (int)(row - last));
        } else {
            w[i] = *reinterpret_cast<const u32_u*>(at + i * ld + voff);
        }
    }
}

// 16 rows of 4 bytes -> 4 columns of 16 bytes
__device__ __forceinline__ void transpose16x4(const uint32_t (&w)[16], v4i (&c)[4]) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const uint32_t t0 = __builtin_amdgcn_perm(w[4 * g + 1], w[4 * g], 0x05010400u), t1 = __builtin_amdgcn_perm(w[4 * g + 1], w[4 * g], 0x07030602u);
        const uint32_t t2 = __builtin_amdgcn_perm(w[4 * g + 3], w[4 * g + 2], 0x05010400u), t3 = __builtin_amdgcn_perm(w[4 * g + 3], w[4 * g + 2], 0x07030602u);
        c[0][g] = (int)__builtin_amdgcn_perm(t2, t0, 0x05040100u);
        c[1][g] = (int)__builtin_amdgcn_perm(t2, t0, 0x07060302u);
        c[2][g] = (int)__builtin_amdgcn_perm(t3, t1, 0x05040100u);
        c[3][g] = (int)__builtin_amdgcn_perm(t3, t1, 0x07060302u);
    }
}

// A lane's four columns of 16 k from the rows: shifted into place where the dwords were read from the end of their rows
// (`ragged`, `flip` are the same in every lane), transposed, sign bits flipped.
template <bool kTail>
__device__ __forceinline__ void columns_of(uint32_t (&w)[16], bool ragged, int shift, uint32_t flip, int k0, int K, v4i (&fb)[4]) {
    if (ragged) {
#pragma unroll
        for (int i = 0; i < 16; ++i) w[i] >>= shift;
    }
    if (flip != 0) {
#pragma unroll
        for (int i = 0; i < 16; ++i)
            if (!kTail || k0 + i < K) w[i] ^= flip;
    }
    transpose16x4(w, fb);
}

// 8 bytes at column `at` of a row of W >= 8, columns outside filled with zp (all of them from W + 8 on)
__device__ __forceinline__ uint64_t window8(const char* row, int at, int W, uint64_t zp) {
    typedef uint64_t u64_u __attribute__((aligned(1)));
    const int from = min(max(at, 0), W - 8), d = at - from, up = min(max(8 * d, 0), 64), down = min(max(-8 * d, 0), 64);
    // (shifts in two halves: 64 is one of the distances)
    const uint64_t v = *reinterpret_cast<const u64_u*>(row + from) ^ zp;
    return ((v >> (up / 2) >> (up - up / 2)) << (down / 2) << (down - down / 2)) ^ zp;
}

__device__ __forceinline__ int32_t sum_bytes(v4i v, int32_t acc) {
#pragma unroll
    for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_sdot4(v[i], 0x01010101, acc, false);
    return acc;
}

}  // namespace
}  // namespace chx
