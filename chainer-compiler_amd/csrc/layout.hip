// Byte-tensor layout changes between NCHW-contiguous arrays (what a caller that knows
// nothing about layouts hands over) and the channels-last layout the MFMA kernels use.
// 64 x 64-byte tiles: a thread brings in four dwords of four rows, transposes the 4 x 4 bytes with eight permutes and
// leaves them in LDS as dwords of the other direction; 16 bytes per lane go out, contiguous along their fastest axis.
// Bound by memory and launch latency; [32, 128, 28, 28] and back around a convolution add 10.4 us to its 9.6, with
// single bytes through LDS 19.6.
#include "conv_mfma.h"
#include "gemm_i8_device.h"

namespace chx {
namespace {

constexpr int kTile = 64, kPitch = 80;  // (rows of LDS: 16-byte aligned)

// The first n of the dword's bytes.
__device__ __forceinline__ uint32_t load_bytes(const uint8_t* p, int n) {
    if (n >= 4) return *reinterpret_cast<const u32_u*>(p);
    uint32_t v = 0;
    for (int i = 0; i < n; ++i) v |= (uint32_t)p[i] << (8 * i);
    return v;
}

// A 64 x 64 tile: `rows` rows of `cols` bytes at src, row pitch src_pitch, become the columns of dst, of which the first
// `cols` rows and `out` bytes (rows and, from there on, zeros) are written.
__device__ __forceinline__ void transpose_tile(const uint8_t* src, int64_t src_pitch, int rows, int cols, uint8_t* dst, int64_t dst_pitch, int out) {
    __shared__ __attribute__((aligned(16))) uint8_t tile[kTile * kPitch];
    const int q = threadIdx.x & 15, r = threadIdx.x >> 4;  // four columns, four rows
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int row = 4 * r + i, left = row < rows ? cols - 4 * q : 0;
        w[i] = load_bytes(src + (int64_t)(row < rows ? row : 0) * src_pitch + 4 * q, left);
    }
    const uint32_t t0 = __builtin_amdgcn_perm(w[1], w[0], 0x05010400u), t1 = __builtin_amdgcn_perm(w[1], w[0], 0x07030602u);
    const uint32_t t2 = __builtin_amdgcn_perm(w[3], w[2], 0x05010400u), t3 = __builtin_amdgcn_perm(w[3], w[2], 0x07030602u);
    const uint32_t c[4] = {__builtin_amdgcn_perm(t2, t0, 0x05040100u), __builtin_amdgcn_perm(t2, t0, 0x07060302u), __builtin_amdgcn_perm(t3, t1, 0x05040100u),
                           __builtin_amdgcn_perm(t3, t1, 0x07060302u)};
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<uint32_t*>(&tile[(4 * q + i) * kPitch + 4 * r]) = c[i];
    __syncthreads();
    const int row = threadIdx.x >> 2, at = (threadIdx.x & 3) * 16, n = out - at;
    if (row >= cols || n <= 0) return;
    const v4i v = *reinterpret_cast<const v4i*>(&tile[row * kPitch + at]);
    uint8_t* d = dst + (int64_t)row * dst_pitch + at;
    if (n >= 16) *reinterpret_cast<v4i_u*>(d) = v;
    else
        for (int i = 0; i < n; ++i) d[i] = tile[row * kPitch + at + i];
}

// src [N][C][HW] -> dst [N][HW][pitch]
__global__ __launch_bounds__(256) void nchw_to_nhwc_u8_kernel(
        const uint8_t* __restrict__ src, uint8_t* __restrict__ dst, int C, int64_t HW, int pitch) {
    const int64_t n = blockIdx.z, p0 = (int64_t)blockIdx.x * kTile;
    const int c0 = blockIdx.y * kTile, cols = (int)(HW - p0 < kTile ? HW - p0 : kTile);
    transpose_tile(src + (n * C + (c0 < C ? c0 : 0)) * HW + p0, HW, min(max(C - c0, 0), kTile), cols, dst + (n * HW + p0) * pitch + c0, pitch, min(pitch - c0, kTile));
}

// src [N][HW][pitch] -> dst [N][C][HW]
__global__ __launch_bounds__(256) void nhwc_to_nchw_u8_kernel(
        const uint8_t* __restrict__ src, uint8_t* __restrict__ dst, int C, int64_t HW, int pitch) {
    const int64_t n = blockIdx.z, p0 = (int64_t)blockIdx.x * kTile;
    const int c0 = blockIdx.y * kTile, rows = (int)(HW - p0 < kTile ? HW - p0 : kTile);
    transpose_tile(src + (n * HW + p0) * pitch + c0, pitch, rows, min(C - c0, kTile), dst + (n * C + c0) * HW + p0, HW, rows);
}

// Channels-last pixels to a pitch of a multiple of 16 bytes; a thread moves 16 of them.  [16, 40, 56, 56] with 120 3x3 filters, packed
// channels-last: 2945 us with one thread per result, 14.0 with this copy in front of the matrix-core kernel.
__global__ __launch_bounds__(256) void pixels_u8_kernel(
        const uint8_t* __restrict__ src, int64_t n_stride, int64_t h_stride, int64_t w_stride, uint8_t* __restrict__ dst, uint32_t total, int C, uint32_t chunks, uint32_t ch_mul, uint32_t ch_shift,
        uint32_t W, uint32_t w_mul, uint32_t w_shift, uint32_t H, uint32_t h_mul, uint32_t h_shift) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= total) return;
    const uint32_t px = (__umulhi(i, ch_mul) + i) >> ch_shift, c = (i - px * chunks) * 16;
    const uint32_t row = (__umulhi(px, w_mul) + px) >> w_shift, w = px - row * W;
    const uint32_t n = (__umulhi(row, h_mul) + row) >> h_shift, h = row - n * H;
    const uint8_t* p = src + (int64_t)n * n_stride + (int64_t)h * h_stride + (int64_t)w * w_stride + c;
    const int left = C - (int)c;
    v4i v;
    if (left >= 16) {
        v = *reinterpret_cast<const v4i_u*>(p);
    } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = (int)load_bytes(p + 4 * k, left - 4 * k);
    }
    reinterpret_cast<v4i*>(dst)[i] = v;
}

}  // namespace

int launch_pixels_u8(const char* src, int64_t n_stride, int64_t h_stride, int64_t w_stride, char* dst, int N, int C, int H, int W, int pitch, hipStream_t s) {
    const int64_t total = (int64_t)N * H * W * (pitch / 16);
    if (total == 0) return CHX_HIP_OK;
    if (total >= (int64_t(1) << 31) - 256) return CHX_HIP_EUNSUPPORTED;
    uint32_t cm, cs, wm, ws, hm, hs;
    magic_divisor((uint32_t)(pitch / 16), &cm, &cs);
    magic_divisor((uint32_t)W, &wm, &ws);
    magic_divisor((uint32_t)H, &hm, &hs);
    pixels_u8_kernel<<<(unsigned)((total + 255) / 256), 256, 0, s>>>(reinterpret_cast<const uint8_t*>(src), n_stride, h_stride, w_stride, reinterpret_cast<uint8_t*>(dst), (uint32_t)total, C,
                                                                    (uint32_t)(pitch / 16), cm, cs, (uint32_t)W, wm, ws, (uint32_t)H, hm, hs);
    return launch_check("pixels_u8_kernel");
}

int launch_nchw_to_nhwc_u8(const char* src, char* dst, int N, int C, int64_t HW, int pitch, hipStream_t s) {
    if (N == 0 || C == 0 || HW == 0) return CHX_HIP_OK;
    dim3 grid((unsigned)((HW + kTile - 1) / kTile), (unsigned)((pitch + kTile - 1) / kTile), (unsigned)N);
    nchw_to_nhwc_u8_kernel<<<grid, 256, 0, s>>>(
            reinterpret_cast<const uint8_t*>(src), reinterpret_cast<uint8_t*>(dst), C, HW, pitch);
    return launch_check("nchw_to_nhwc_u8_kernel");
}

int launch_nhwc_to_nchw_u8(const char* src, char* dst, int N, int C, int64_t HW, int pitch, hipStream_t s) {
    if (N == 0 || C == 0 || HW == 0) return CHX_HIP_OK;
    dim3 grid((unsigned)((HW + kTile - 1) / kTile), (unsigned)((C + kTile - 1) / kTile), (unsigned)N);
    nhwc_to_nchw_u8_kernel<<<grid, 256, 0, s>>>(
            reinterpret_cast<const uint8_t*>(src), reinterpret_cast<uint8_t*>(dst), C, HW, pitch);
    return launch_check("nhwc_to_nchw_u8_kernel");
}

}  // namespace chx
