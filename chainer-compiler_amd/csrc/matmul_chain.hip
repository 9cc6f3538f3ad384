// A chain of quantized matrix products, the layers of a multi-layer perceptron, as one launch:
//
//   [QuantizeLinear] -> QLinearMatMul -> ... -> QLinearMatMul -> [DequantizeLinear]
//
// Bound by latency: a layer of such a network is a few hundred nanoseconds of loads and products, but as a launch of its
// own 3.5 to 4 us with the hand-over from the kernel before it, and its host side another 2.5.  Here a work-group takes
// 16 rows through all layers: the codes between them stay in LDS, and the weights of a layer are requested before the sums of
// the layer before it are requantized, so that only the first layer waits for memory.  784 -> 100 -> 100 -> 10 over 32 rows
// 17.0 -> 8.5 us, Program.run of it, with the result on the host, 27-31 -> 19.5.
//
// The weights are laid out once, as fragments of v_mfma_i32_16x16x64_i8 (1 KB for 64 k of 16 columns, a lane's 16 bytes
// together), zeros where a matrix ends, and behind them the sum of each column: read as they lie, a step took 100
// instructions for their transposition instead of 10, and a layer of 512 x 512 8 us instead of 3.5.  The sixteen wavefronts
// share out columns and K and add their sums in LDS, in int32, so that the order does not matter.  Every quantization is
// the reference's, operation by operation: the codes are those of the single ops.
#include <cstring>

#include "contract.h"
#include "conv_device.h"
#include "gemm_i8_device.h"

struct chx_hip_chain_weights {
    char* fragments = nullptr;
    int32_t K = 0, N = 0;
    int32_t is_signed = 0;
    int device = 0;
};

namespace chx {
namespace {

constexpr int kWaves = 16, kRows = 16;
// (the codes and sums of a work-group then are 49.7 KB, below the 64 KB that a kernel has without asking; 1024 columns would be 82 KB)
constexpr int kMaxLayers = 6, kMaxK = 1024, kMaxN = 512;
constexpr int kActRow = kMaxK + 16, kSumRow = kMaxN + 4;  // (off a multiple of the LDS banks)
constexpr int kDepth = 8;                                 // fragments of weights in flight per wavefront

struct ChainLayer {
    const char* b;         // fragments, then the columns' sums (int32, a whole number of fragments' columns)
    int32_t N, K, steps;   // steps: fragments along K
    int32_t tiles, tiles_inverse, slices, per;  // columns in tiles of 16; see part_of
    int32_t ca, cb;        // what is left of the zero points when the codes are read as signed bytes (gemm_i8.hip)
    uint32_t y_flip;       // of the layer's codes where they stay in LDS: 0x80808080 for unsigned ones
    float scale;           // of the sums
    QuantParams q;
    float inv_scale;
};

struct ChainArgs {
    ChainLayer layer[kMaxLayers];
    const char* x;
    int64_t x_row;
    int32_t x_is_float;
    uint32_t x_flip;
    QuantParams xq;
    float x_inv_scale, x_largest;  // 1 / scale; 2^40 scale
    char* y;
    int64_t y_row;
    int32_t y_is_float;
    float y_zpf, y_scale;
    int32_t M, layers;
};

// the dword's bytes from `valid` on zero
__device__ __forceinline__ uint32_t keep_bytes(uint32_t v, int valid) {
    return valid >= 4 ? v : valid <= 0 ? 0 : v & ((1u << (8 * valid)) - 1);
}

// quantize_value with its division in three instructions: what saturates anyway is limited first, so that no intermediate
// leaves the range of float32 (NaN goes the way of the largest value, as it does there).
__device__ __forceinline__ int32_t quantize_any(float v, const QuantParams& q, float inv_scale, float largest) {
    v = v < largest ? v : largest;
    return quantize_value_folded<false>(__builtin_fmaxf(v, -largest), q, inv_scale, q.lo);
}

__global__ __launch_bounds__(64 * kWaves) void matmul_chain_kernel(ChainArgs) {
    __shared__ __attribute__((aligned(16))) char act[kRows * kActRow];    // codes as signed bytes, zeros up to a multiple of 64
    __shared__ __attribute__((aligned(16))) int32_t sum[kRows * kSumRow];  // 0 between layers
    const ChainArgs& g = kernel_arguments<ChainArgs>();
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15, group = lane >> 4;
    const int m0 = (int)blockIdx.x * kRows;

    // This wavefront's part of a layer: `count` fragments from `at` on, the first of them step `first` of column tile `tile`.
    // With fewer than sixteen tiles it is a slice of the steps of one (w / tiles = w * tiles_inverse >> 8 for w < 16), with
    // more it is all steps of `per` of them.
    struct Part {
        const v4i* at;
        int count, tile, first, end;  // end: of the tile's steps
    };
    auto part_of = [&](const ChainLayer& L) __attribute__((always_inline)) {
        Part p;
        if (L.slices > 1) {
            const int slice = wave * L.tiles_inverse >> 8;
            p.tile = wave - slice * L.tiles;
            p.first = min(slice * L.per, L.steps);
            p.end = slice < L.slices ? min(p.first + L.per, L.steps) : p.first;
            p.count = p.end - p.first;
        } else {
            p.tile = min(wave * L.per, L.tiles);
            p.first = 0;
            p.end = L.steps;
            p.count = min(L.per, L.tiles - p.tile) * L.steps;
        }
        p.at = reinterpret_cast<const v4i*>(L.b) + (p.tile * L.steps + p.first) * 64 + lane;
        return p;
    };
    v4i ring[kDepth];
    Part p = part_of(g.layer[0]);
    // (past the end of a wavefront's fragments the last one again: no branch around a load)
    auto load_first = [&]() __attribute__((always_inline)) {
        if (p.count > 0) {
#pragma unroll
            for (int d = 0; d < kDepth; ++d) ring[d] = p.at[min(d, p.count - 1) * 64];
        }
    };
    load_first();

    // the input: a row per wavefront
    {
        const int K = g.layer[0].K, row = min(m0 + wave, g.M - 1), padded = g.layer[0].steps * 64;
        const char* x = g.x + (int64_t)row * g.x_row;
        if (g.x_is_float) {
            typedef float v4f_u __attribute__((ext_vector_type(4), aligned(4)));
            const float* xf = reinterpret_cast<const float*>(x);
            v4f_u v[kMaxK / 256];
#pragma unroll
            for (int i = 0; i < kMaxK / 256; ++i) {
                const int k = 256 * i + 4 * lane;
                v[i] = v4f_u{0.f, 0.f, 0.f, 0.f};
                if (k + 4 <= K) v[i] = *reinterpret_cast<const v4f_u*>(xf + k);
                else
                    for (int e = 0; e < 3; ++e)
                        if (k + e < K) v[i][e] = xf[k + e];
            }
            for (int i = threadIdx.x; i < kRows * kSumRow / 4; i += 64 * kWaves) reinterpret_cast<v4i*>(sum)[i] = v4i{0, 0, 0, 0};
#pragma unroll
            for (int i = 0; i < kMaxK / 256; ++i) {
                const int k = 256 * i + 4 * lane;
                if (256 * i >= padded) break;
                int32_t code[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) code[e] = quantize_any(v[i][e], g.xq, g.x_inv_scale, g.x_largest);
                const uint32_t word = pack4(code[0], code[1], code[2], code[3]);
                if (k < padded) *reinterpret_cast<uint32_t*>(act + wave * kActRow + k) = keep_bytes(word ^ g.x_flip, K - k);
            }
        } else {
            for (int i = threadIdx.x; i < kRows * kSumRow / 4; i += 64 * kWaves) reinterpret_cast<v4i*>(sum)[i] = v4i{0, 0, 0, 0};
            for (int k = lane; k < padded; k += 64) act[wave * kActRow + k] = k < K ? (char)(x[k] ^ (char)g.x_flip) : (char)0;
        }
    }
    __syncthreads();

    for (int l = 0; l < g.layers; ++l) {
        const ChainLayer& L = g.layer[l];
        // the columns' sums that this thread's codes take, before anything is waited for (asked for where they are used, behind the barrier,
        // they are a memory latency per layer: 8.9 us for 8.5 at 784 -> 100 -> 100 -> 10 over 32 rows)
        const v4i* columns = reinterpret_cast<const v4i*>(L.b + (int64_t)L.tiles * L.steps * 1024);
        v4i of_column[kMaxN / 256];
#pragma unroll
        for (int i = 0; i < kMaxN / 256; ++i) of_column[i] = columns[min(lane + 64 * i, L.tiles * 4 - 1)];
        if (p.count > 0) {
            v4i acc = {0, 0, 0, 0};
            int step = p.first, tile = p.tile;
            const char* a = act + col * kActRow + group * 16;
            auto multiply = [&](v4i b) __attribute__((always_inline)) {
                acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(*reinterpret_cast<const v4i*>(a + step * 64), b, acc, 0, 0, 0);
                if (++step == p.end) {
                    // (columns from N on are added too, to places that the next layer's codes take as zeros)
#pragma unroll
                    for (int r = 0; r < 4; ++r) atomicAdd(&sum[(group * 4 + r) * kSumRow + tile * 16 + col], acc[r]);
                    acc = v4i{0, 0, 0, 0};
                    step = 0;
                    ++tile;
                }
            };
            int f = 0;
            for (; f + kDepth < p.count; f += kDepth) {
#pragma unroll
                for (int d = 0; d < kDepth; ++d) {
                    multiply(ring[d]);
                    ring[d] = p.at[min(f + d + kDepth, p.count - 1) * 64];
                }
            }
#pragma unroll
            for (int d = 0; d < kDepth; ++d)
                if (f + d < p.count) multiply(ring[d]);
        }
        const bool last = l + 1 == g.layers;
        // the zero points' share: of a row here, of the columns below
        int32_t of_row = 0;
        if (L.cb != 0) {
            int32_t s = 0;
            for (int k = 4 * lane; k < L.steps * 64; k += 256) s = __builtin_amdgcn_sdot4(*reinterpret_cast<const int32_t*>(act + wave * kActRow + k), 0x01010101, s, false);
#pragma unroll
            for (int d = 1; d < 64; d *= 2) s += __shfl_xor(s, d);
            of_row = L.cb * (s + L.K * L.ca);
        }
        if (!last) {
            p = part_of(g.layer[l + 1]);
            load_first();
        }
        __syncthreads();
        const int padded = last ? L.tiles * 16 : (L.tiles + 3) / 4 * 64;
#pragma unroll
        for (int i = 0; i < kMaxN / 256; ++i) {
            const int n = 4 * lane + 256 * i;
            if (n >= padded) break;
            v4i* at = reinterpret_cast<v4i*>(&sum[wave * kSumRow + n]);
            v4i v = *at + of_row;
            if (n < L.N) v += L.ca * of_column[i];
            int32_t code[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) code[e] = quantize_value_folded<false>((float)v[e] * L.scale, L.q, L.inv_scale, L.q.lo);
            if (!last) {
                *at = v4i{0, 0, 0, 0};
                *reinterpret_cast<uint32_t*>(act + wave * kActRow + n) = keep_bytes(pack4(code[0], code[1], code[2], code[3]) ^ L.y_flip, L.N - n);
            } else if (m0 + wave < g.M) {
                char* y = g.y + (int64_t)(m0 + wave) * g.y_row;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (n + e >= L.N) continue;
                    if (g.y_is_float) reinterpret_cast<float*>(y)[n + e] = dequantize_value(code[e], g.y_zpf, g.y_scale);
                    else y[n + e] = (char)code[e];
                }
            }
        }
        if (!last) __syncthreads();
    }
}

// A work-group per column tile: its fragments, a wavefront each in turn, and the sums of its columns.
__global__ __launch_bounds__(256) void chain_weights_kernel(const uint8_t* b, int64_t row, int64_t column, int32_t K, int32_t N, uint32_t flip, char* out) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, steps = (K + 63) / 64, tile = (int)blockIdx.x;
    const int n = tile * 16 + (lane & 15);
    __shared__ int32_t sums[16];
    if (threadIdx.x < 16) sums[threadIdx.x] = 0;
    __syncthreads();
    int32_t sum = 0;
    for (int s = wave; s < steps; s += 4) {
        v4i v = {0, 0, 0, 0};
        for (int i = 0; i < 16; ++i) {
            const int k = s * 64 + (lane >> 4) * 16 + i;
            if (n < N && k < K) v[i / 4] |= (int)((uint32_t)(uint8_t)(b[k * row + n * column] ^ flip) << (8 * (i % 4)));
        }
        sum = sum_bytes(v, sum);
        *reinterpret_cast<v4i*>(out + ((int64_t)(tile * steps + s) * 64 + lane) * 16) = v;
    }
    atomicAdd(&sums[lane & 15], sum);
    __syncthreads();
    if (threadIdx.x < 16) reinterpret_cast<int32_t*>(out + (int64_t)gridDim.x * steps * 1024)[tile * 16 + threadIdx.x] = sums[threadIdx.x];
}

bool zero_point_fits(int32_t zp, int32_t dtype) {
    return dtype == CHX_HIP_INT8 ? zp >= -128 && zp <= 127 : zp >= 0 && zp <= 255;
}

// rows one behind the other, elements of a row next to each other
bool is_rows(const chx_hip_tensor& t) {
    const int64_t es = dtype_size(t.dtype);
    return t.ndim == 2 && (t.shape[1] == 1 || t.strides[1] == es) && t.strides[0] >= 0 && t.strides[0] % es == 0 && aligned(t.data, (size_t)es);
}

// Above 8192 rows every compute unit has a third work-group to begin with, and narrow layers are faster as launches that fill the
// chip at once.  Both times in us, fitted to 305 networks of one to six layers, 8 to 512 columns and 4,096 to 16,384 rows, measured both ways inside
// a recording (within 5 and 12 %).  All of them as chains were 0.82 of the time of single calls on average, but 28 slower by more than 5 %
// (15797 x 1005 -> 32 -> 107 codes 23.2 and 34.6 us, 16033 x 148 -> 44 -> 44 20.4 and 25.2); by this choice 0.84, and by at most 5 %.
bool slower_in_rounds(const ChainArgs& g) {
    if (g.M <= 8192) return false;
    const double rounds = (double)((g.M + 256 * kRows - 1) / (256 * kRows)), million_rows = 1e-6 * g.M;
    const int32_t K = g.layer[0].K, N = g.layer[g.layers - 1].N;
    double chain = 0.47 + (g.x_is_float ? 0.615 * ((K + 255) / 256) : 0.149 * ((K + 63) / 64));
    double single = (g.x_is_float + g.y_is_float) * 2.82 + million_rows * (0.49 * K + (g.x_is_float ? 0.80 * K : 0.0) + (g.y_is_float ? 0.12 * N : 0.0));
    for (int i = 0; i < g.layers; ++i) {
        const ChainLayer& L = g.layer[i];
        chain += 0.342 + 0.085 * (L.slices > 1 ? L.per : L.per * L.steps) + 0.943 * ((L.N + 255) / 256);
        single += 4.45 + million_rows * (3.68e-3 * L.K * L.N + 1.69 * L.N);
    }
    return 3.44 + rounds * chain + 0.308 * million_rows * N * (g.y_is_float ? 4 : 1) > 0.9 * single;
}

}  // namespace
}  // namespace chx

using namespace chx;

extern "C" int chx_hip_chain_weights_create(const chx_hip_tensor* b, void* stream, chx_hip_chain_weights** out) {
    CHX_REQUIRE(out != nullptr, "chain weights: null output");
    *out = nullptr;
    CHX_PROPAGATE(check_tensor(b, "chain weights"));
    CHX_REQUIRE(is_q8(b->dtype), "chain weights: uint8 or int8, got %s", dtype_name(b->dtype));
    if (b->ndim != 2 || b->shape[0] < 1 || b->shape[0] > kMaxK || b->shape[1] < 1 || b->shape[1] > kMaxN) CHX_FAIL(CHX_HIP_EUNSUPPORTED, "chain weights: a matrix of at most %d x %d", kMaxK, kMaxN);
    const int64_t steps = (b->shape[0] + 63) / 64, tiles = (b->shape[1] + 15) / 16;
    chx_hip_chain_weights w;
    CHX_HIP_CALL(hipGetDevice(&w.device));
    void* p = nullptr;
    CHX_PROPAGATE(spare_memory(&p, (size_t)(tiles * steps * 1024 + tiles * 64), "chain weights"));
    w.fragments = static_cast<char*>(p);
    w.K = (int32_t)b->shape[0];
    w.N = (int32_t)b->shape[1];
    w.is_signed = b->dtype == CHX_HIP_INT8;
    chain_weights_kernel<<<(unsigned)tiles, 256, 0, as_stream(stream)>>>(
            static_cast<const uint8_t*>(b->data), b->strides[0], b->strides[1], w.K, w.N, w.is_signed ? 0u : 0x80u, w.fragments);
    int rc = launch_check("chain_weights_kernel");
    // (later calls may come on any stream)
    if (rc == CHX_HIP_OK && hipStreamSynchronize(as_stream(stream)) != hipSuccess) {
        set_error("chain weights: the stream is in error");
        rc = CHX_HIP_ERUNTIME;
    }
    if (rc != CHX_HIP_OK) {
        (void)hipFree(p);
        return rc;
    }
    *out = new chx_hip_chain_weights(w);
    return CHX_HIP_OK;
}

extern "C" void chx_hip_chain_weights_destroy(chx_hip_chain_weights* w) {
    if (!w) return;
    (void)hipFree(w->fragments);
    delete w;
}

extern "C" int chx_hip_qlinear_chain(
        const chx_hip_tensor* x, float x_scale, int32_t x_zero_point, int32_t x_dtype, const chx_hip_chain_layer* layers, int32_t n,
        chx_hip_tensor* y, float y_scale, int32_t y_zero_point, void* stream) {
    CHX_PROPAGATE(check_tensor(x, "chain x"));
    CHX_PROPAGATE(check_tensor(y, "chain y"));
    CHX_REQUIRE(layers != nullptr && n >= 1, "chain: no layers");
    auto refuse = [](const char* why) {
        set_error("chain of products: %s", why);
        return (int)CHX_HIP_EUNSUPPORTED;
    };
    if (n > kMaxLayers) return refuse("too many layers");
    if (!is_rows(*x) || !is_rows(*y) || x->shape[0] < 1) return refuse("operands that are not rows");
    // One work-group a compute unit up to 4096 rows; one after the other beyond.  us for the whole network on this kernel / as single
    // calls, by rows:                         32             256            4096           16384
    //    784 -> 100 -> 100 -> 10            8.9 / 17.0      9.0 / 17.8     9.3 / 22.8    33.0 / 37.2
    //    1024 -> 512 -> 512 -> 100         13.5 / 17.8     13.7 / 18.9    16.3 / 34.1    57.2 / 65.4
    //    1024 -> 512                        9.7 / 10.9      9.9 / 11.1    13.5 / 21.0    45.5 / 46.7
    //    six layers of 512                 22.7 / 30.8     22.9 / 32.6    26.8 / 53.4    92.9 / 115
    // (and see slower_in_rounds)
    if (x->shape[0] > 16384) return refuse("too many rows");
    int device = 0;
    CHX_HIP_CALL(hipGetDevice(&device));
    ChainArgs g;
    memset(&g, 0, sizeof(g));
    g.x_is_float = x->dtype == CHX_HIP_FLOAT32;
    if (!g.x_is_float && x->dtype != x_dtype) return refuse("the type of x");
    if (!is_q8(x_dtype) || !zero_point_fits(x_zero_point, x_dtype)) return refuse("the quantization of x");
    g.x = static_cast<const char*>(x->data);
    g.x_row = x->strides[0];
    g.M = (int32_t)x->shape[0];
    if (g.x_is_float && !(x_scale > 1e-20f && x_scale < 1e20f)) return refuse("the scale of x");
    g.xq = make_quant_params(x_scale, x_zero_point, x_dtype == CHX_HIP_INT8);
    g.x_inv_scale = 1.0f / x_scale;
    g.x_largest = 0x1p40f * x_scale;
    g.x_flip = x_dtype == CHX_HIP_UINT8 ? 0x80808080u : 0;
    int64_t k = x->shape[1];
    int32_t dtype = x_dtype;
    for (int i = 0; i < n; ++i) {
        const chx_hip_chain_layer& in = layers[i];
        ChainLayer& L = g.layer[i];
        if (in.b == nullptr || in.b->device != device) return refuse("a layer's weights");
        if (in.b->K != k || (i > 0 && k > kMaxN)) return refuse("a layer's size");
        if (!is_q8(in.y_dtype) || !zero_point_fits(in.a_zero_point, dtype) || !zero_point_fits(in.b_zero_point, in.b->is_signed ? CHX_HIP_INT8 : CHX_HIP_UINT8) || !zero_point_fits(in.y_zero_point, in.y_dtype))
            return refuse("a layer's quantization");
        // no intermediate of the short division may leave the range of float32 (the same bounds as in gemm_i8.hip)
        const double largest = 0x1p31 * fabs((double)in.a_scale * (double)in.b_scale);
        if (!(in.y_scale > 1e-20f && in.y_scale < 1e20f && largest < 1e30 && largest / (double)in.y_scale < 1e30)) return refuse("a layer's scales");
        L.b = in.b->fragments;
        L.K = in.b->K;
        L.N = in.b->N;
        L.steps = (L.K + 63) / 64;
        L.tiles = (L.N + 15) / 16;
        L.tiles_inverse = (255 + L.tiles) / L.tiles;
        L.slices = L.tiles < kWaves ? kWaves / L.tiles : 1;
        L.per = L.slices > 1 ? (L.steps + L.slices - 1) / L.slices : (L.tiles + kWaves - 1) / kWaves;
        L.ca = (dtype == CHX_HIP_UINT8 ? 128 : 0) - in.a_zero_point;
        L.cb = (in.b->is_signed ? 0 : 128) - in.b_zero_point;
        L.y_flip = in.y_dtype == CHX_HIP_UINT8 ? 0x80808080u : 0;
        L.scale = in.a_scale * in.b_scale;
        L.q = make_quant_params(in.y_scale, in.y_zero_point, in.y_dtype == CHX_HIP_INT8);
        L.inv_scale = 1.0f / in.y_scale;
        k = L.N;
        dtype = in.y_dtype;
    }
    g.layers = n;
    if (y->shape[0] != x->shape[0] || y->shape[1] != k) return refuse("the shape of y");
    g.y_is_float = y->dtype == CHX_HIP_FLOAT32;
    if (!g.y_is_float && y->dtype != dtype) return refuse("the type of y");
    g.y = static_cast<char*>(y->data);
    g.y_row = y->strides[0];
    g.y_zpf = (float)y_zero_point;
    g.y_scale = y_scale;
    if (slower_in_rounds(g)) return refuse("slower than its layers for so many rows");
    matmul_chain_kernel<<<(unsigned)((g.M + kRows - 1) / kRows), 64 * kWaves, 0, as_stream(stream)>>>(g);
    return launch_check("matmul_chain_kernel");
}
