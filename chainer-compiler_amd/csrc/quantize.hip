// QuantizeLinear / DequantizeLinear for gfx950: one pass over HBM, 128-bit loads and
// stores, no temporaries.  Arithmetic follows quantize_array / dequantize_array of the
// reference (runtime/ops/quantize.cc:16-44) operation by operation in fp32; the file is
// compiled with -ffp-contract=off so no multiply-add is fused.
#include "chx_internal.h"
#include "quant_math.h"

namespace chx {
namespace {

constexpr int kThreads = 256;

typedef float v4f __attribute__((ext_vector_type(4)));
// the same for views that start anywhere: one access each all the same
typedef float v4f_u __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32_u __attribute__((aligned(1)));

// One 128-bit load and one 32-bit store per lane and step, kUnroll steps per thread at
// a stride of one block, so that every access instruction of a wavefront covers one
// contiguous span (1 KiB in, 256 B out).
constexpr int kUnroll = 4;
// QuantizeLinear of a tensor of a few million elements (a network's input) is a launch of some 10 us, bound by how
// many wavefronts issue at once rather than by bytes in flight: one step per thread then (10.3 against 11.5 us for
// [64, 3, 224, 224]); four steps are 4 % faster on [64, 1024, 1024].
constexpr int64_t kFewVectors = int64_t(1) << 22;

// The up to three elements behind the last vector go with the thread that would have had the next one: a launch of their
// own took 2 to 3 us of the 7 of a small tensor.
template <bool kRne, int kSteps>
__global__ __launch_bounds__(kThreads) void quantize_flat_kernel(const float* __restrict__ x, uint8_t* __restrict__ y, int64_t n, QuantParams qp) {
    const int64_t first = (int64_t)blockIdx.x * (kThreads * kSteps) + threadIdx.x, n_vec = n / 4;
    v4f v[kSteps];
#pragma unroll
    for (int u = 0; u < kSteps; ++u) {
        const int64_t i = first + u * kThreads;
        if (i < n_vec) v[u] = __builtin_nontemporal_load(reinterpret_cast<const v4f_u*>(x) + i);
    }
#pragma unroll
    for (int u = 0; u < kSteps; ++u) {
        const int64_t i = first + u * kThreads;
        if (i < n_vec) {
            const uint32_t out = pack4(quantize_value<kRne>(v[u].x, qp), quantize_value<kRne>(v[u].y, qp),
                                       quantize_value<kRne>(v[u].z, qp), quantize_value<kRne>(v[u].w, qp));
            __builtin_nontemporal_store(out, reinterpret_cast<u32_u*>(y) + i);
        } else if (i == n_vec) {
            for (int64_t e = 4 * n_vec; e < n; ++e) y[e] = (uint8_t)quantize_value<kRne>(x[e], qp);
        }
    }
}

__device__ __forceinline__ int64_t strided_offset(int64_t flat, const StridedDesc& d) {
    int64_t off = 0;
    for (int a = d.ndim - 1; a >= 0; --a) {
        const int64_t q = flat / d.shape[a];
        const int64_t r = flat - q * d.shape[a];
        off += r * d.strides[a];
        flat = q;
    }
    return off;
}

// Any strides on either side (element [i0,i1,..] of x goes to element [i0,i1,..] of y).
template <bool kRne>
__global__ __launch_bounds__(kThreads) void quantize_strided_kernel(
        const char* __restrict__ x, StridedDesc xd, char* __restrict__ y, StridedDesc yd, int64_t n, QuantParams qp) {
    const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (i >= n) return;
    const float v = *reinterpret_cast<const float*>(x + strided_offset(i, xd));
    *reinterpret_cast<uint8_t*>(y + strided_offset(i, yd)) = (uint8_t)quantize_value<kRne>(v, qp);
}

template <bool kSigned>
__device__ __forceinline__ v4f dequant4(uint32_t w, float zpf, float scale) {
    v4f r;
    r.x = dequantize_value(byte_of<kSigned>(w, 0), zpf, scale);
    r.y = dequantize_value(byte_of<kSigned>(w, 1), zpf, scale);
    r.z = dequantize_value(byte_of<kSigned>(w, 2), zpf, scale);
    r.w = dequantize_value(byte_of<kSigned>(w, 3), zpf, scale);
    return r;
}

template <bool kSigned, int kSteps>
__global__ __launch_bounds__(kThreads) void dequantize_flat_kernel(const uint8_t* __restrict__ x, float* __restrict__ y, int64_t n, float zpf, float scale) {
    const int64_t first = (int64_t)blockIdx.x * (kThreads * kSteps) + threadIdx.x, n_vec = n / 4;
    uint32_t q[kSteps];
#pragma unroll
    for (int u = 0; u < kSteps; ++u) {
        const int64_t i = first + u * kThreads;
        if (i < n_vec) q[u] = __builtin_nontemporal_load(reinterpret_cast<const u32_u*>(x) + i);
    }
#pragma unroll
    for (int u = 0; u < kSteps; ++u) {
        const int64_t i = first + u * kThreads;
        if (i < n_vec) {
            const v4f v = dequant4<kSigned>(q[u], zpf, scale);
            __builtin_nontemporal_store(v, reinterpret_cast<v4f_u*>(y) + i);
        } else if (i == n_vec) {
            for (int64_t e = 4 * n_vec; e < n; ++e) y[e] = dequantize_value(kSigned ? (int32_t)(int8_t)x[e] : (int32_t)x[e], zpf, scale);
        }
    }
}

template <bool kSigned>
__global__ __launch_bounds__(kThreads) void dequantize_strided_kernel(
        const char* __restrict__ x, StridedDesc xd, char* __restrict__ y, StridedDesc yd, int64_t n, float zpf,
        float scale) {
    const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (i >= n) return;
    const uint8_t raw = *reinterpret_cast<const uint8_t*>(x + strided_offset(i, xd));
    const int32_t q = kSigned ? (int32_t)(int8_t)raw : (int32_t)raw;
    *reinterpret_cast<float*>(y + strided_offset(i, yd)) = dequantize_value(q, zpf, scale);
}

inline unsigned blocks_for(int64_t n) {
    return (unsigned)((n + kThreads - 1) / kThreads);
}

inline unsigned flat_blocks_for(int64_t n, int steps) {
    const int64_t threads = n / 4 + (n % 4 != 0 ? 1 : 0);
    return (unsigned)((threads + kThreads * steps - 1) / (kThreads * steps));
}

StridedDesc make_desc(const chx_hip_tensor& t) {
    StridedDesc d;
    d.ndim = t.ndim;
    for (int i = 0; i < t.ndim; ++i) {
        d.shape[i] = t.shape[i];
        d.strides[i] = t.strides[i];
    }
    return d;
}

}  // namespace
}  // namespace chx

using namespace chx;

extern "C" int chx_hip_quantize_linear(
        const chx_hip_tensor* x, float y_scale, int32_t y_zero_point, uint32_t flags, chx_hip_tensor* y, void* stream) {
    CHX_PROPAGATE(check_tensor(x, "QuantizeLinear x"));
    CHX_PROPAGATE(check_tensor(y, "QuantizeLinear y"));
    CHX_REQUIRE(x->dtype == CHX_HIP_FLOAT32, "QuantizeLinear: x must be float32, got %s", dtype_name(x->dtype));
    CHX_REQUIRE(is_q8(y->dtype), "QuantizeLinear: y must be uint8 or int8, got %s", dtype_name(y->dtype));
    CHX_REQUIRE(same_shape(*x, *y), "QuantizeLinear: x and y shapes differ");
    const bool i8 = y->dtype == CHX_HIP_INT8;
    // CHECK_LE(min, zp) / CHECK_LE(zp, max), runtime/ops/quantize.cc:26-27
    CHX_REQUIRE(y_zero_point >= (i8 ? -128 : 0) && y_zero_point <= (i8 ? 127 : 255),
                "QuantizeLinear: zero point %d outside the range of %s", y_zero_point, dtype_name(y->dtype));
    const int64_t n = numel(*x);
    if (n == 0) return CHX_HIP_OK;
    CHX_REQUIRE(n < (int64_t(1) << 40), "QuantizeLinear: %lld elements is beyond what one launch covers", (long long)n);
    const bool rne = (flags & CHX_HIP_ROUND_ONNX_RNE) != 0;
    QuantParams qp = make_quant_params(y_scale, y_zero_point, i8);
    hipStream_t s = as_stream(stream);

    if (same_dense_layout(*x, *y)) {
        const float* xp = static_cast<const float*>(x->data);
        uint8_t* yp = static_cast<uint8_t*>(y->data);
#define CHX_QUANTIZE(RNE, STEPS) quantize_flat_kernel<RNE, STEPS><<<flat_blocks_for(n, STEPS), kThreads, 0, s>>>(xp, yp, n, qp)
        if (n / 4 <= kFewVectors) {
            if (rne) CHX_QUANTIZE(true, 1);
            else CHX_QUANTIZE(false, 1);
        } else {
            if (rne) CHX_QUANTIZE(true, kUnroll);
            else CHX_QUANTIZE(false, kUnroll);
        }
#undef CHX_QUANTIZE
        return launch_check("quantize_flat_kernel");
    }
    const StridedDesc xd = make_desc(*x), yd = make_desc(*y);
    if (rne)
        quantize_strided_kernel<true><<<blocks_for(n), kThreads, 0, s>>>(
                static_cast<const char*>(x->data), xd, static_cast<char*>(y->data), yd, n, qp);
    else
        quantize_strided_kernel<false><<<blocks_for(n), kThreads, 0, s>>>(
                static_cast<const char*>(x->data), xd, static_cast<char*>(y->data), yd, n, qp);
    return launch_check("quantize_strided_kernel");
}

extern "C" int chx_hip_dequantize_linear(
        const chx_hip_tensor* x, float x_scale, int32_t x_zero_point, chx_hip_tensor* y, void* stream) {
    CHX_PROPAGATE(check_tensor(x, "DequantizeLinear x"));
    CHX_PROPAGATE(check_tensor(y, "DequantizeLinear y"));
    CHX_REQUIRE(is_q8(x->dtype), "DequantizeLinear: x must be uint8 or int8, got %s", dtype_name(x->dtype));
    CHX_REQUIRE(y->dtype == CHX_HIP_FLOAT32, "DequantizeLinear: y must be float32, got %s", dtype_name(y->dtype));
    CHX_REQUIRE(same_shape(*x, *y), "DequantizeLinear: x and y shapes differ");
    const int64_t n = numel(*x);
    if (n == 0) return CHX_HIP_OK;
    CHX_REQUIRE(n < (int64_t(1) << 40), "DequantizeLinear: %lld elements is beyond what one launch covers", (long long)n);
    const bool i8 = x->dtype == CHX_HIP_INT8;
    const float zpf = (float)x_zero_point;
    hipStream_t s = as_stream(stream);

    if (same_dense_layout(*x, *y)) {
        const uint8_t* xp = static_cast<const uint8_t*>(x->data);
        float* yp = static_cast<float*>(y->data);
#define CHX_DEQUANTIZE(SIGNED, STEPS) dequantize_flat_kernel<SIGNED, STEPS><<<flat_blocks_for(n, STEPS), kThreads, 0, s>>>(xp, yp, n, zpf, x_scale)
        if (n / 4 <= kFewVectors) {
            if (i8) CHX_DEQUANTIZE(true, 1);
            else CHX_DEQUANTIZE(false, 1);
        } else {
            if (i8) CHX_DEQUANTIZE(true, kUnroll);
            else CHX_DEQUANTIZE(false, kUnroll);
        }
#undef CHX_DEQUANTIZE
        return launch_check("dequantize_flat_kernel");
    }
    const StridedDesc xd = make_desc(*x), yd = make_desc(*y);
    if (i8)
        dequantize_strided_kernel<true><<<blocks_for(n), kThreads, 0, s>>>(
                static_cast<const char*>(x->data), xd, static_cast<char*>(y->data), yd, n, zpf, x_scale);
    else
        dequantize_strided_kernel<false><<<blocks_for(n), kThreads, 0, s>>>(
                static_cast<const char*>(x->data), xd, static_cast<char*>(y->data), yd, n, zpf, x_scale);
    return launch_check("dequantize_strided_kernel");
}
