// Entry points of the integer contractions: QLinearConv, ConvInteger, MatMulInteger,
// QLinearMatMul.  Validation and shape rules follow the reference's RunImpl bodies
// (runtime/ops/quantize.cc:62-146) and GroupedConv (runtime/chainerx_util.cc:313-340);
// the arithmetic is in the kernels.
#include <algorithm>
#include <array>
#include <climits>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "contract.h"
#include "conv_mfma.h"
#include "inverted_residual.h"
#include "bottleneck.h"
#include "depthwise.h"

namespace chx {
namespace {

struct ConvShape {
    int32_t N, C, H, W, OC, Cg, KH, KW, OH, OW;
};

int conv_shape(
        const chx_hip_tensor& x, const chx_hip_tensor& w, const chx_hip_conv_params& p, const chx_hip_tensor& y,
        const char* op, ConvShape* cs) {
    CHX_REQUIRE(x.ndim == 4 && w.ndim == 4 && y.ndim == 4, "%s: x, w and y must be 4-D (2-D convolution only)", op);
    CHX_REQUIRE(is_q8(x.dtype), "%s: x must be uint8 or int8, got %s", op, dtype_name(x.dtype));
    CHX_REQUIRE(is_q8(w.dtype), "%s: w must be uint8 or int8, got %s", op, dtype_name(w.dtype));
    CHX_REQUIRE(p.group >= 1 && p.stride_h >= 1 && p.stride_w >= 1, "%s: group and strides must be positive", op);
    CHX_REQUIRE(p.pad_h_begin >= 0 && p.pad_w_begin >= 0 && p.pad_h_end >= 0 && p.pad_w_end >= 0,
                "%s: negative padding is not supported", op);
    for (int i = 0; i < 4; ++i)
        CHX_REQUIRE(x.shape[i] <= INT32_MAX && w.shape[i] <= INT32_MAX, "%s: extent too large", op);
    cs->N = (int32_t)x.shape[0];
    cs->C = (int32_t)x.shape[1];
    cs->H = (int32_t)x.shape[2];
    cs->W = (int32_t)x.shape[3];
    cs->OC = (int32_t)w.shape[0];
    cs->Cg = (int32_t)w.shape[1];
    cs->KH = (int32_t)w.shape[2];
    cs->KW = (int32_t)w.shape[3];
    CHX_REQUIRE(cs->C == cs->Cg * p.group, "%s: x has %d channels but w expects %d x group %d", op, cs->C, cs->Cg, p.group);
    CHX_REQUIRE(cs->OC % p.group == 0, "%s: %d output channels do not divide into %d groups", op, cs->OC, p.group);
    const int64_t eh = (int64_t)cs->H + p.pad_h_begin + p.pad_h_end - cs->KH;
    const int64_t ew = (int64_t)cs->W + p.pad_w_begin + p.pad_w_end - cs->KW;
    CHX_REQUIRE(eh >= 0 && ew >= 0, "%s: kernel %dx%d larger than the padded input", op, cs->KH, cs->KW);
    cs->OH = (int32_t)(eh / p.stride_h + 1);
    cs->OW = (int32_t)(ew / p.stride_w + 1);
    CHX_REQUIRE(y.shape[0] == cs->N && y.shape[1] == cs->OC && y.shape[2] == cs->OH && y.shape[3] == cs->OW,
                "%s: y is [%lld,%lld,%lld,%lld], expected [%d,%d,%d,%d]", op, (long long)y.shape[0], (long long)y.shape[1],
                (long long)y.shape[2], (long long)y.shape[3], cs->N, cs->OC, cs->OH, cs->OW);
    return CHX_HIP_OK;
}

// A 0-d or 1-d parameter array with `expect_one_or` elements.
int param_vector(const chx_hip_tensor& t, int64_t per_channel, const char* what, int64_t* len, int64_t* stride) {
    CHX_REQUIRE(t.ndim <= 1, "%s must be 0-d or 1-d", what);
    *len = numel(t);
    CHX_REQUIRE(*len == 1 || *len == per_channel, "%s has %lld elements, expected 1 or %lld", what, (long long)*len,
                (long long)per_channel);
    *stride = t.ndim == 1 ? t.strides[0] : 0;
    return CHX_HIP_OK;
}

void fill_conv_args(
        const chx_hip_tensor& x, const chx_hip_tensor& w, const chx_hip_conv_params& p, const chx_hip_tensor& y,
        const ConvShape& cs, ConvDirectArgs* a) {
    memset(a, 0, sizeof(*a));
    a->x = static_cast<const char*>(x.data);
    a->w = static_cast<const char*>(w.data);
    a->y = static_cast<char*>(y.data);
    for (int i = 0; i < 4; ++i) {
        a->xs[i] = x.strides[i];
        a->ws[i] = w.strides[i];
        a->ys[i] = y.strides[i];
    }
    a->N = cs.N; a->C = cs.C; a->H = cs.H; a->W = cs.W;
    a->OC = cs.OC; a->Cg = cs.Cg; a->KH = cs.KH; a->KW = cs.KW; a->OH = cs.OH; a->OW = cs.OW;
    a->sh = p.stride_h; a->sw = p.stride_w; a->ph = p.pad_h_begin; a->pw = p.pad_w_begin; a->group = p.group;
    a->x_signed = x.dtype == CHX_HIP_INT8;
    a->w_signed = w.dtype == CHX_HIP_INT8;
    a->total = (int64_t)cs.N * cs.OC * cs.OH * cs.OW;
    a->D = a->KD = a->OD = a->sd = 1;  // no third spatial axis
}

int fill_requant(
        float x_scale, float y_scale, int32_t y_zp, const chx_hip_tensor& y, const chx_hip_tensor* bias, int64_t bias_len,
        uint32_t flags, const char* op, RequantParams* rq, const int32_t** bias_ptr) {
    CHX_REQUIRE(is_q8(y.dtype), "%s: y must be uint8 or int8, got %s", op, dtype_name(y.dtype));
    const bool i8 = y.dtype == CHX_HIP_INT8;
    CHX_REQUIRE(y_zp >= (i8 ? -128 : 0) && y_zp <= (i8 ? 127 : 255), "%s: zero point %d outside the range of %s", op,
                y_zp, dtype_name(y.dtype));
    rq->q = make_quant_params(y_scale, y_zp, i8);
    rq->x_scale = x_scale;
    rq->relu_floor = (flags & CHX_HIP_FUSE_RELU) ? y_zp : INT32_MIN;
    rq->bias_mode = kBiasNone;
    *bias_ptr = nullptr;
    if (bias) {
        CHX_PROPAGATE(check_tensor(bias, "bias"));
        CHX_REQUIRE(bias->dtype == CHX_HIP_INT32, "%s: bias must be int32, got %s", op, dtype_name(bias->dtype));
        CHX_REQUIRE(bias->ndim == 1 && bias->shape[0] == bias_len && is_contiguous(*bias),
                    "%s: bias must be a contiguous [%lld] vector", op, (long long)bias_len);
        rq->bias_mode = (flags & CHX_HIP_BIAS_ONNX_INT32) ? kBiasOnnxInt32 : kBiasReferenceFloat;
        *bias_ptr = static_cast<const int32_t*>(bias->data);
    }
    return CHX_HIP_OK;
}

struct MatMulShape {
    int64_t batch, M, K, N;
    int64_t a_batch, b_batch, y_batch;
};

// NumpyMatMul, runtime/chainerx_util.cc:210-230: 2-D Dot, or N-D with equal leading dims
// flattened into a batch.  Leading dims must be contiguous among themselves.
int matmul_shape(const chx_hip_tensor& a, const chx_hip_tensor& b, const chx_hip_tensor& y, const char* op, MatMulShape* ms) {
    CHX_REQUIRE(a.ndim >= 2 && b.ndim == a.ndim && y.ndim == a.ndim, "%s: a, b and y must have the same ndim >= 2", op);
    const int nd = a.ndim;
    ms->M = a.shape[nd - 2];
    ms->K = a.shape[nd - 1];
    ms->N = b.shape[nd - 1];
    CHX_REQUIRE(b.shape[nd - 2] == ms->K, "%s: inner dimensions differ (%lld vs %lld)", op, (long long)ms->K,
                (long long)b.shape[nd - 2]);
    CHX_REQUIRE(y.shape[nd - 2] == ms->M && y.shape[nd - 1] == ms->N, "%s: y has the wrong matrix shape", op);
    ms->batch = 1;
    for (int i = 0; i < nd - 2; ++i) {
        CHX_REQUIRE(a.shape[i] == b.shape[i] && a.shape[i] == y.shape[i], "%s: leading dimensions differ", op);
        ms->batch *= a.shape[i];
    }
    auto batch_stride = [&](const chx_hip_tensor& t, int64_t* out) -> int {
        // leading axes must collapse into one
        *out = 0;
        int64_t expect = -1;
        for (int i = nd - 3; i >= 0; --i) {
            if (t.shape[i] == 1) continue;
            if (expect < 0) {
                *out = t.strides[i];
                expect = t.strides[i] * t.shape[i];
            } else {
                CHX_REQUIRE(t.strides[i] == expect, "%s: leading dimensions are not collapsible", op);
                expect *= t.shape[i];
            }
        }
        return CHX_HIP_OK;
    };
    CHX_PROPAGATE(batch_stride(a, &ms->a_batch));
    CHX_PROPAGATE(batch_stride(b, &ms->b_batch));
    CHX_PROPAGATE(batch_stride(y, &ms->y_batch));
    return CHX_HIP_OK;
}

void fill_matmul_args(
        const chx_hip_tensor& a, const chx_hip_tensor& b, const chx_hip_tensor& y, const MatMulShape& ms, MatMulDirectArgs* m) {
    memset(m, 0, sizeof(*m));
    const int nd = a.ndim;
    m->a = static_cast<const char*>(a.data);
    m->b = static_cast<const char*>(b.data);
    m->y = static_cast<char*>(y.data);
    m->a_batch = ms.a_batch; m->a_row = a.strides[nd - 2]; m->a_col = a.strides[nd - 1];
    m->b_batch = ms.b_batch; m->b_row = b.strides[nd - 2]; m->b_col = b.strides[nd - 1];
    m->y_batch = ms.y_batch; m->y_row = y.strides[nd - 2]; m->y_col = y.strides[nd - 1];
    m->M = ms.M; m->K = ms.K; m->N = ms.N;
    m->total = ms.batch * ms.M * ms.N;
    m->a_signed = a.dtype == CHX_HIP_INT8;
    m->b_signed = b.dtype == CHX_HIP_INT8;
}


// ---- MFMA path -------------------------------------------------------------------------------

inline int round_up(int v, int m) {
    return (v + m - 1) / m * m;
}

// Packed weights for the MFMA kernel (see conv_mfma.hip).
struct PackedWeights {
    int8_t* wp = nullptr;       // and in the same allocation the others, but for
    int8_t* wf_apart = nullptr;  // wf, where that has one of its own
    int32_t* wsum = nullptr;
    int32_t* padsum = nullptr;  // ConvMfmaArgs::padsum, null for dense packing and for more than 32 taps
    int C64 = 0, OCpad = 0, KP = 0;
    int BK = 64;         // K bytes per kernel step; the packed layout depends on it
    bool dense = false;  // taps packed densely; activations go through an explicit im2col
    int8_t* wf = nullptr;  // of a plan with at most 32 taps: the weights in the order of the small tiles
    int8_t* wd = nullptr;  // dense only: the same weights in the order of the planar-input kernel
};

// Dense packing pays when per-tap padding to 64 channels would at least double the K extent, and the channels do not fill
// 16 bytes: from there on the pixels are read as they are and the zero products cost less than the expanded matrix
// ([64, 16, 56, 56] with 16 3x3 filters: 45.3 us expanded, 16.9 this way).
bool prefer_dense(int C, int KH, int KW) {
    return C < 16 && KH * KW > 1 && round_up(C, 64) * KH * KW >= 2 * round_up(C * KH * KW, 64);
}

size_t packed_bytes(int OC, int C, int KH, int KW, PackedWeights* pw) {
    pw->OCpad = round_up(OC, 128);
    pw->dense = prefer_dense(C, KH, KW);
    if (pw->dense) {
        pw->KP = round_up(C * KH * KW, 64);
        pw->C64 = pw->KP;
    } else {
        pw->C64 = round_up(C, 64);
        pw->KP = KH * KW * pw->C64;
    }
    // whole cache lines per pixel and step when the channels allow it
    pw->BK = (!pw->dense && pw->C64 % 128 == 0) ? 128 : 64;
    return (size_t)pw->OCpad * pw->KP;
}

// The weights qualify for the MFMA kernel: one group, int8, accumulator cannot overflow.
bool weights_fit_mfma(const chx_hip_tensor& w, int group) {
    if (group != 1 || w.dtype != CHX_HIP_INT8) return false;
    if (w.shape[1] > (1 << 20) || w.shape[2] * w.shape[3] > 64) return false;  // one mask bit per filter tap
    PackedWeights pw;
    packed_bytes(1, (int)w.shape[1], (int)w.shape[2], (int)w.shape[3], &pw);
    return (int64_t)pw.KP * 128 * 128 < (int64_t(1) << 31) && w.shape[0] < (1 << 24);
}

// How a convolution is launched, beyond what its operands decide.  The defaults are what a host wants; the
// environment variables are overrides for tuning and for tests (which reach every launch configuration through them),
// read when a plan is created or a one-shot entry point is called, never on the path of a plan's runs.
//   CHX_HIP_TILE=<oc>,<px>[,<work-groups per compute unit>[,<wavefronts: 4 or 8>]]  forces a launch configuration (with the
//                               small tiles, in place of the work-groups: 1 for pixels from LDS, where that fits; 100 for the tiles
//                               of conv_same_kernel)
//   CHX_HIP_AUTOTUNE=0          keeps the heuristic tile choice instead of timing the configurations
//   CHX_HIP_NO_STEM=1           keeps few-channel first layers off the planar-input kernel
//   CHX_HIP_AFFINE_RESIDUAL=0   keeps fused residual sums on the operation-by-operation arithmetic
struct LaunchOptions {
    bool forced_tile = false;
    int tile_oc = 0, tile_px = 0, max_wgs_per_cu = 0, waves = 4;
    bool autotune = true;
    bool stem_kernel = true;
    bool affine_residual = true;
};

LaunchOptions read_launch_options() {
    LaunchOptions o;
    if (const char* env = getenv("CHX_HIP_TILE")) {
        int toc = 0, tpx = 0, cap = 0, wv = 4;
        const int got = sscanf(env, "%d,%d,%d,%d", &toc, &tpx, &cap, &wv);
        if (got >= 2 && cap >= 0) {
            o.forced_tile = true;
            o.tile_oc = toc;
            o.tile_px = tpx;
            o.max_wgs_per_cu = got >= 3 ? cap : 0;
            o.waves = wv;
            o.autotune = false;
        }
    }
    if (const char* e = getenv("CHX_HIP_AUTOTUNE")) o.autotune = o.autotune && e[0] != '0';
    o.stem_kernel = getenv("CHX_HIP_NO_STEM") == nullptr;
    if (const char* e = getenv("CHX_HIP_AFFINE_RESIDUAL")) o.affine_residual = e[0] != '0';
    return o;
}

// Tile shape: the largest tile that still gives every compute unit a work-group.
void pick_tile(const LaunchOptions& opt, const ConvMfmaArgs& a, bool out_int32, int* tile_oc, int* tile_px, int* max_wgs_per_cu, int* waves) {
    *waves = 4;
    if (opt.forced_tile) {
        const int toc = opt.tile_oc, tpx = opt.tile_px, wv = opt.waves;
        const bool same = opt.max_wgs_per_cu == kConvSame;
        const bool four = wv == 4 && (toc == 64 || toc == 128) && (tpx == 64 || tpx == 128);
        const bool eight = wv == 8 && ((toc == 128 && tpx == 128) || (a.bk == 128 && ((toc == 128 && tpx == 256) || (toc == 64 && tpx == 128))));
        if (same ? conv_same_has(toc, tpx, wv) && conv_same_takes(a, tpx) && !out_int32 : four || eight || (conv_split_has(toc, tpx, wv) && conv_split_takes(a) && !out_int32) ||
            (toc == kConvPointTile.oc && tpx == kConvPointTile.px && wv == kConvPointTile.waves && conv_point_takes(a) && !out_int32)) {
            *tile_oc = toc;
            *tile_px = tpx;
            *max_wgs_per_cu = opt.max_wgs_per_cu;
            *waves = wv;
            return;
        }
    }
    static const int cand[4][2] = {{128, 128}, {64, 128}, {128, 64}, {64, 64}};
    const int64_t want = 256;
    for (int i = 0; i < 4; ++i) {
        int toc = cand[i][0], tpx = cand[i][1];
        if (a.OC <= 64 && toc > 64) continue;
        const int64_t blocks = (int64_t)((a.OC + toc - 1) / toc) * ((a.M + tpx - 1) / tpx);
        *tile_oc = toc;
        *tile_px = tpx;
        if (blocks >= want) return;
    }
}

// Launch configurations measured for the input shapes a plan has seen: the first eager call on
// a new shape times the tile shapes and occupancy caps on the call's own operands (every
// configuration writes the same bytes) and later calls reuse the fastest.
struct TunedConfig {
    int64_t M;
    int32_t H, W, OH, OW;
    int64_t x_n_stride, x_h_stride, x_w_stride;  // a kernel may take a dense image only (conv_point_takes)
    bool short_form;                             // ... or a requantization in a short form only (conv_same_takes)
    int tile_oc, tile_px, max_wgs_per_cu;
    int waves;      // wavefronts per work-group
    bool with_res;  // measured with a fused residual sum (an entry of its own: the epilogue differs)
    int32_t oc_split = 0;  // measured as two convolutions in one launch, split here (restricts the tiles)
};
struct TuneCache {
    std::vector<TunedConfig> entries;
};

struct Configuration {
    int tile_oc, tile_px, max_wgs_per_cu, waves;
};

// What was measured for one plan holds for every other one of the same geometry: a network repeats most of its
// convolutions, and a second program over the same shapes finds all of them measured.
class MeasuredConfigurations {
public:
    using Key = std::array<int64_t, 25>;
    static Key key(const ConvMfmaArgs& a, bool xu, bool out_int32, bool rne) {
        int device = 0;
        (void)hipGetDevice(&device);
        const int64_t res = a.res.r ? 1 + a.res.affine : 0;
        return {device, a.M, a.H, a.W, a.OH, a.OW, a.KH, a.KW, a.sh, a.sw, a.ph, a.pw, a.C16, a.KP, a.bk, a.OC, a.oc_split, a.x_n_stride,
                a.x_h_stride, a.x_w_stride, a.y_px_stride, aligned(a.y, 16), res, (a.x_zp & 0xff) != 0, (xu ? 1 : 0) | (out_int32 ? 2 : 0) | (rne ? 4 : 0) | (a.qp.path != 0 ? 8 : 0)};
    }
    bool find(const Key& k, Configuration* c) {
        std::lock_guard<std::mutex> lock(mutex_);
        const auto it = known_.find(k);
        if (it == known_.end()) return false;
        *c = it->second;
        return true;
    }
    void add(const Key& k, const Configuration& c) {
        std::lock_guard<std::mutex> lock(mutex_);
        if (known_.size() >= 4096) known_.clear();  // bounded: a program of ever new shapes measures again
        known_[k] = c;
    }

private:
    std::mutex mutex_;
    std::map<Key, Configuration> known_;
};

MeasuredConfigurations& measured_configurations() {
    static MeasuredConfigurations* m = new MeasuredConfigurations;
    return *m;
}

constexpr size_t kReadThrough = size_t(64) << 20;  // twice the L2 caches of the device's 8 XCDs

// Times the launch configurations on the call's operands and gives the fastest.
int tune_conv_mfma(const ConvMfmaArgs& a, bool xu, bool out_int32, bool rne, hipStream_t s, Configuration* best) {
    // tile (output channels x pixels), wavefronts; the eight-wavefront kernels take the compute unit alone
    static const int tiles[7][3] = {{128, 128, 4}, {64, 128, 4}, {128, 64, 4}, {64, 64, 4}, {128, 128, 8}, {128, 256, 8}, {64, 128, 8}};
    struct Candidate {
        Configuration c;
        std::vector<float> seen;
        float ms() const {  // the median
            std::vector<float> v = seen;
            std::sort(v.begin(), v.end());
            return v.empty() ? 1e30f : v[v.size() / 2];
        }
    };
    std::vector<Candidate> all;
    for (const auto& t : tiles) {
        if (a.OC <= 64 && t[0] > 64) continue;
        if (a.oc_split % t[0] != 0) continue;  // two outputs: a tile belongs to one of them whole (floats: none of these)
        if (t[2] == 8 && (t[0] == 64 || t[1] == 256) && a.bk != 128) continue;
        const int64_t tiles_all = (int64_t)((a.OC + t[0] - 1) / t[0]) * ((a.M + t[1] - 1) / t[1]);
        all.push_back({{t[0], t[1], 0, t[2]}, {}});
        // (a cap that the tiles do not reach is the launch without one)
        if (t[2] == 4 && tiles_all > 512) all.push_back({{t[0], t[1], 2, t[2]}, {}});
        if (t[2] == 4 && tiles_all > 256) all.push_back({{t[0], t[1], 1, t[2]}, {}});
    }
    // launches that the staged tiles fill (in tiles of 64 x 64, eight per compute unit) are not for the small tiles: they
    // read their operands from L2 once per tile
    if (!out_int32 && conv_split_takes(a) && (int64_t)((a.OC + 63) / 64) * ((a.M + 63) / 64) <= 2048)
        for (const ConvSplitTile& t : kConvSplitTiles)
            if (t.waves * 512 / t.oc <= a.KP) {  // (half a step and more for every wavefront)
                all.push_back({{t.oc, t.px, 0, t.waves}, {}});
                if (conv_split_patch_takes(a, t.oc, t.px, t.waves)) all.push_back({{t.oc, t.px, kConvSplitPatch, t.waves}, {}});
            }

    if (!out_int32 && !rne)
        for (const ConvSplitTile& t : kConvSameTiles)
            if (conv_same_takes(a, t.px) && (a.OC > 64 || t.oc == 64)) all.push_back({{t.oc, t.px, kConvSame, t.waves}, {}});
    if (!out_int32 && a.oc_split != kFloatResults && conv_point_takes(a))
        for (int per_cu : {2, 4, 6}) all.push_back({{kConvPointTile.oc, kConvPointTile.px, per_cu, kConvPointTile.waves}, {}});

    std::vector<hipEvent_t> events(2 * all.size());
    size_t created = 0;
    int rc = CHX_HIP_OK;
    while (created < events.size() && hipEventCreate(&events[created]) == hipSuccess) ++created;
    if (created < events.size()) rc = CHX_HIP_ERUNTIME;
    void* other = nullptr;
    if (rc == CHX_HIP_OK && hipMallocAsync(&other, kReadThrough, s) != hipSuccess) {
        (void)hipGetLastError();
        other = nullptr;  // (no memory to spare: the first look's verdict stands)
    }
    auto launch = [&](const Configuration& c) {
        if (rc == CHX_HIP_OK) rc = launch_conv_mfma(a, c.tile_oc, c.tile_px, c.max_wgs_per_cu, c.waves, xu, out_int32, rne, s);
    };
    // every candidate once: `times` launches in a row after one that warms up, or one that finds the L2 caches full of
    // something else; one wait for all of them
    auto look = [&](int times, bool cold) {
        for (size_t i = 0; i < all.size() && rc == CHX_HIP_OK; ++i) {
            if (cold) rc = launch_read_through(other, kReadThrough, s);
            else launch(all[i].c);
            if (rc == CHX_HIP_OK && hipEventRecord(events[2 * i], s) != hipSuccess) rc = CHX_HIP_ERUNTIME;
            for (int t = 0; t < times; ++t) launch(all[i].c);
            if (rc == CHX_HIP_OK && hipEventRecord(events[2 * i + 1], s) != hipSuccess) rc = CHX_HIP_ERUNTIME;
        }
        if (rc == CHX_HIP_OK && hipStreamSynchronize(s) != hipSuccess) rc = CHX_HIP_ERUNTIME;
        for (size_t i = 0; i < all.size() && rc == CHX_HIP_OK; ++i) {
            float ms = 0.f;
            if (hipEventElapsedTime(&ms, events[2 * i], events[2 * i + 1]) != hipSuccess) rc = CHX_HIP_ERUNTIME;
            all[i].seen.push_back(ms / times);
        }
    };
    auto faster = [](const Candidate& l, const Candidate& r) { return l.ms() < r.ms(); };
    // Two launches in a row each, to find the eight worth a closer look.  Those again, one launch at a time with cold
    // caches: in a network a layer's weights and the previous layer's results come from memory, and a configuration that
    // reads them in many places loses there what it wins in a loop (512 -> 128 channels of 8 images of 28 x 28: 12 us in the
    // network with the tile that a loop prefers, 6 with another).
    look(2, false);
    std::sort(all.begin(), all.end(), faster);
    if (all.size() > 8) all.resize(8);
    if (other) {
        for (Candidate& c : all) c.seen.clear();
        for (int round = 0; round < 5; ++round) look(1, true);
        (void)hipFreeAsync(other, s);
    }
    for (size_t i = 0; i < created; ++i) (void)hipEventDestroy(events[i]);
    if (rc != CHX_HIP_OK) CHX_FAIL(rc, "timing the convolution launch configurations failed: %s", chx_hip_last_error());
    *best = std::min_element(all.begin(), all.end(), faster)->c;
    return CHX_HIP_OK;
}

struct XLayout {
    const char* ptr;
    int64_t n_stride, h_stride, w_stride;
    bool direct;  // usable as is
};

// channels-last view with 16-byte aligned pixels whose pitch covers round_up(C, 16) bytes
bool x_is_mfma_ready(const chx_hip_tensor& x) {
    const int64_t C = x.shape[1];
    if (C != 1 && x.strides[1] != 1) return false;
    const int64_t c16 = (C + 15) / 16 * 16;
    if (!aligned(x.data, 16)) return false;
    for (int ax : {0, 2, 3}) {
        if (x.shape[ax] == 1) continue;
        if (x.strides[ax] % 16 != 0 || x.strides[ax] < c16) return false;
    }
    // reading c16 bytes of the last pixel must stay inside the allocation: guaranteed when every
    // pixel pitch covers c16 bytes, which the loop above checked for all axes of extent > 1
    if (x.shape[3] == 1 && x.shape[2] == 1 && x.shape[0] == 1) return C == c16;
    return true;
}

// pixel-major output: (n, oh, ow) collapse to one index with a single stride, channels unit stride
bool y_is_pixel_major(const chx_hip_tensor& y, int64_t* px_stride) {
    const int64_t es = dtype_size(y.dtype);
    if (y.shape[1] != 1 && y.strides[1] != es) return false;
    int64_t stride = -1, expect = -1;
    for (int ax : {3, 2, 0}) {
        if (y.shape[ax] == 1) continue;
        if (stride < 0) {
            stride = y.strides[ax];
            expect = stride * y.shape[ax];
        } else {
            if (y.strides[ax] != expect) return false;
            expect *= y.shape[ax];
        }
    }
    if (stride < 0) stride = y.shape[1] * es;
    if (stride < y.shape[1] * es) return false;
    *px_stride = stride;
    return true;
}

// [lowest, highest + 1) byte address any element of t occupies
void byte_range(const chx_hip_tensor& t, uintptr_t* lo, uintptr_t* hi) {
    int64_t below = 0, above = dtype_size(t.dtype);
    for (int i = 0; i < t.ndim; ++i) {
        if (t.shape[i] <= 1) continue;
        const int64_t span = (t.shape[i] - 1) * t.strides[i];
        if (span < 0) below += span;
        else above += span;
    }
    *lo = reinterpret_cast<uintptr_t>(t.data) + below;
    *hi = reinterpret_cast<uintptr_t>(t.data) + above;
}

bool byte_ranges_overlap(const chx_hip_tensor& a, const chx_hip_tensor& b) {
    if (numel(a) == 0 || numel(b) == 0) return false;
    uintptr_t alo, ahi, blo, bhi;
    byte_range(a, &alo, &ahi);
    byte_range(b, &blo, &bhi);
    return alo < bhi && blo < ahi;
}

// Scratch buffers that outlive a call: a plan keeps its transposition / im2col space so that
// repeated runs allocate nothing (and can be captured into a HIP graph).  Grow-only.
struct ScratchCache {
    void* ptr[2] = {nullptr, nullptr};
    size_t size[2] = {0, 0};
    bool pinned = false;  // a recorded run holds these addresses: the buffers must not move
};

struct ConvCall {
    TuneCache* tune;      // null: heuristic tile choice
    ScratchCache* cache;  // null: stream-ordered scratch for this call only
    const chx_hip_tensor* x;
    chx_hip_tensor* y;
    const chx_hip_conv_params* p;
    ConvShape cs;
    int32_t x_zp;
    bool out_int32;
    bool rne;
    const float* w_scale;
    int32_t w_scale_len;
    const int32_t* bias;
    RequantParams rq;
    const ResidualAdd* res = nullptr;  // a residual sum fused behind the requantization
    LaunchOptions opt;                 // the plan's, or read for this one-shot call
    // two convolutions of x in one launch (ConvMfmaArgs::oc_split): the second one's output and requantization
    const chx_hip_tensor* y2 = nullptr;
    int32_t oc_split = 0;
    RequantParams rq2;
    // CHX_HIP_STORE_MINUS_128 for y / y2: the stored byte is the uint8 code minus 128
    bool y_minus_128 = false, y2_minus_128 = false;
    // x's values before their QuantizeLinear, which the kernel does on the way (x then only describes the codes)
    const chx_hip_tensor* x_float = nullptr;
    QuantProduct xq = {};
    // where the result goes as floats (y then only describes its codes)
    float* dq = nullptr;
    int64_t dq_px = 0;
    float dq_zpf = 0.f, dq_scale = 0.f;
};

// Runs the MFMA kernel on packed weights.  x may be channels-last (used in place) or
// NCHW-contiguous (transposed into scratch first); y may be pixel-major (written in place) or
// NCHW-contiguous 8-bit (written to scratch, then transposed).  Returns EUNSUPPORTED when the
// operand layouts fit neither, so that the caller can fall back to the direct kernel.
int acquire_scratch(ScratchCache* cache, int slot, size_t bytes, hipStream_t s, void** out) {
    if (!cache) return scratch_alloc(out, bytes, s);
    if (cache->size[slot] < bytes) {
        if (cache->pinned)
            CHX_FAIL(CHX_HIP_EPINNED,
                     "this convolution plan is pinned by a recorded run and would have to move its scratch memory (%zu bytes needed, %zu held): "
                     "run larger inputs before recording, or after the recording has been destroyed", bytes, cache->size[slot]);
        // the old buffer may still be in use by work queued on the stream
        CHX_HIP_CALL(hipStreamSynchronize(s));
        if (cache->ptr[slot]) CHX_HIP_CALL(hipFree(cache->ptr[slot]));
        cache->ptr[slot] = nullptr;
        cache->size[slot] = 0;
        CHX_HIP_CALL(hipMalloc(&cache->ptr[slot], bytes));
        cache->size[slot] = bytes;
    }
    *out = cache->ptr[slot];
    return CHX_HIP_OK;
}

void release_scratch(ScratchCache* cache, void* p, hipStream_t s) {
    if (!cache) scratch_free(p, s);
}

int run_conv_mfma(const ConvCall& c, const PackedWeights& pw, hipStream_t s) {
    const chx_hip_tensor& x = *c.x;
    chx_hip_tensor& y = *c.y;
    const ConvShape& cs = c.cs;
    const int C16 = round_up(cs.C, 16);
    void* x_scratch = nullptr;
    void* y_scratch = nullptr;
    ConvMfmaArgs a;
    memset(&a, 0, sizeof(a));
    int KH = cs.KH, KW = cs.KW, H = cs.H, W = cs.W, sh = c.p->stride_h, sw = c.p->stride_w, ph = c.p->pad_h_begin,
        pw_ = c.p->pad_w_begin, C16eff = C16;
    // few channels read from planar rows: the direct kernel, no expanded matrix
    const bool stem = pw.dense && pw.wd && !c.out_int32 && x.strides[3] == 1 &&
                      stem_patch_fits(cs.C, cs.KH, cs.KW, sh, sw) && ph < 64 && pw_ < 64 &&
                      (int64_t)cs.C * (x.strides[1] < 0 ? -x.strides[1] : x.strides[1]) < (int64_t(1) << 30) &&
                      x.strides[2] > 0 && (int64_t)cs.H * x.strides[2] < (int64_t(1) << 30) && c.opt.stem_kernel;
    if (c.x_float) {
        // (the kernel's offsets inside an image are 32 bits, those of floats four times the codes')
        const int64_t channels = (int64_t)cs.C * c.x_float->strides[1], rows = (int64_t)cs.H * c.x_float->strides[2], most = int64_t(1) << 30;
        if (channels <= -most || channels >= most || rows >= most || cs.W >= most / 4) CHX_FAIL(CHX_HIP_EUNSUPPORTED, "QuantizeLinear and QLinearConv as one launch: an image of 1 GB");
        if (!stem || c.rne || cs.W < 4 || !stem_patch_is_small(cs.C, cs.KH, cs.KW, sh, sw, pw_))
            CHX_FAIL(CHX_HIP_EUNSUPPORTED, "QuantizeLinear and QLinearConv as one launch: few channels in planar rows and small filters only");
    }
    // ... from the first row of a tile's to the last, also of those outside the image; a distance between rows that a single one does not have is not
    // counted (launch below).  What lies further apart is left to the direct kernel, which needs no scratch memory either.
    if (stem && cs.H > 1) {
        const chx_hip_tensor& values = c.x_float ? *c.x_float : x;
        const int64_t channels = (int64_t)cs.C * (values.strides[1] < 0 ? -values.strides[1] : values.strides[1]);
        if (stem_patch_rows(cs.KH, sh) * values.strides[2] + channels >= (int64_t(1) << 32)) CHX_FAIL(CHX_HIP_EUNSUPPORTED, "the planar-input kernel: rows too far apart");
    }
    // Channels-last pixels at another pitch than 16 bytes (40 channels packed, say) are copied to one.  The copy's memory is
    // this call's and not the plan's: the direct kernel, which has always taken such arrays, lets one plan run on two streams
    // and inside a recording, pinned or not, and needs none.  A recording keeps that kernel (its memory would have to
    // outlive the call), and so does a pair, which is refused here.
    const bool pixels_copied = !stem && !pw.dense && !x_is_mfma_ready(x) && !is_contiguous(x) && x.strides[1] == 1;
    ScratchCache own;
    Scratch own_memory;
    ScratchCache* cache = pixels_copied ? &own : c.cache;
    if (pixels_copied) {
        if (c.y2 || stream_is_capturing(s)) CHX_FAIL(CHX_HIP_EUNSUPPORTED, "QLinearConv: packed pixels are not copied for a pair or inside a recording");
        int64_t y_px = 0;
        own.size[0] = ((size_t)cs.N * cs.H * cs.W * C16 + 255) / 256 * 256;
        own.size[1] = y_is_pixel_major(y, &y_px) ? 0 : (size_t)cs.N * cs.OH * cs.OW * round_up(cs.OC, 16);
        CHX_PROPAGATE(own_memory.acquire(own.size[0] + own.size[1], s));
        own.ptr[0] = own_memory.ptr();
        own.ptr[1] = static_cast<char*>(own_memory.ptr()) + own.size[0];
    }
    if (c.dq && (stem || pw.dense || !x_is_mfma_ready(x) || c.out_int32 || c.res || c.y2)) CHX_FAIL(CHX_HIP_EUNSUPPORTED, "QLinearConv+DequantizeLinear: channels-last arrays of at least 16 channels only");
    if (stem && c.res) CHX_FAIL(CHX_HIP_EUNSUPPORTED, "the planar-input kernel has no fused residual sum");
    if (stem) {
        // x is used in place
    } else if (pw.dense) {
        // explicit im2col: [M][Kd] bytes, then a 1x1 convolution over Kd channels and M pixels in a row
        const int64_t M = (int64_t)cs.N * cs.OH * cs.OW;
        CHX_REQUIRE(M <= INT32_MAX, "QLinearConv: too many output pixels for the im2col path");
        CHX_PROPAGATE(acquire_scratch(cache, 0, (size_t)M * pw.KP, s, &x_scratch));
        Im2colArgs ia;
        memset(&ia, 0, sizeof(ia));
        ia.x = static_cast<const char*>(x.data);
        for (int i = 0; i < 4; ++i) ia.xs[i] = x.strides[i];
        ia.C = cs.C; ia.H = cs.H; ia.W = cs.W; ia.OH = cs.OH; ia.OW = cs.OW; ia.KH = cs.KH; ia.KW = cs.KW;
        ia.sh = sh; ia.sw = sw; ia.ph = ph; ia.pw = pw_;
        ia.Kd = pw.KP;
        ia.fill = c.x_zp;
        ia.M = M;
        ia.col = static_cast<char*>(x_scratch);
        const int rc = launch_im2col_dense(ia, s);
        if (rc != CHX_HIP_OK) {
            release_scratch(cache, x_scratch, s);
            return rc;
        }
        a.x = static_cast<const char*>(x_scratch);
        a.x_w_stride = pw.KP;
        a.x_h_stride = 0;
        a.x_n_stride = 0;
        KH = KW = 1; H = 1; W = (int)M; sh = sw = 1; ph = pw_ = 0;
        C16eff = pw.KP;
    } else if (x_is_mfma_ready(x)) {
        a.x = static_cast<const char*>(x.data);
        a.x_n_stride = x.strides[0];
        a.x_h_stride = x.strides[2];
        a.x_w_stride = x.strides[3];
    } else if (is_contiguous(x) || pixels_copied) {
        const int64_t HW = (int64_t)cs.H * cs.W;
        CHX_PROPAGATE(acquire_scratch(cache, 0, (size_t)cs.N * HW * C16, s, &x_scratch));
        const int rc_x = is_contiguous(x) ? launch_nchw_to_nhwc_u8(static_cast<const char*>(x.data), static_cast<char*>(x_scratch), cs.N, cs.C, HW, C16, s)
                                          : launch_pixels_u8(static_cast<const char*>(x.data), x.strides[0], x.strides[2], x.strides[3], static_cast<char*>(x_scratch), cs.N, cs.C, cs.H, cs.W, C16, s);
        if (rc_x != CHX_HIP_OK) {
            release_scratch(cache, x_scratch, s);
            return rc_x;
        }
        a.x = static_cast<const char*>(x_scratch);
        a.x_w_stride = C16;
        a.x_h_stride = (int64_t)cs.W * C16;
        a.x_n_stride = HW * C16;
    } else {
        CHX_FAIL(CHX_HIP_EUNSUPPORTED, "x layout is neither channels-last nor NCHW-contiguous");
    }
    const int64_t es = c.out_int32 ? 4 : 1;
    int64_t y_px = 0;
    bool y_post = false;
    if (y_is_pixel_major(y, &y_px)) {
        a.y = static_cast<char*>(y.data);
        a.y_px_stride = y_px;
    } else if (is_contiguous(y) && !c.out_int32 && !c.res) {
        const int64_t OHW = (int64_t)cs.OH * cs.OW;
        const int pitch = round_up(cs.OC, 16);
        const int rc_y = acquire_scratch(cache, 1, (size_t)cs.N * OHW * pitch, s, &y_scratch);
        if (rc_y != CHX_HIP_OK) {
            release_scratch(cache, x_scratch, s);
            return rc_y;
        }
        a.y = static_cast<char*>(y_scratch);
        a.y_px_stride = pitch;
        y_post = true;
    } else {
        release_scratch(cache, x_scratch, s);
        CHX_FAIL(CHX_HIP_EUNSUPPORTED, "y layout is neither pixel-major nor NCHW-contiguous 8-bit");
    }
    (void)es;
    if (c.y_minus_128 || c.y2_minus_128) {
        if (stem || y_post || c.out_int32) {
            release_scratch(cache, x_scratch, s);
            release_scratch(cache, y_scratch, s);
            CHX_FAIL(CHX_HIP_EUNSUPPORTED, "QLinearConv: codes minus 128 are stored by the matrix-core kernel into channels-last results only");
        }
        a.y_flip = c.y_minus_128 ? 0x80808080u : 0u;
    }
    if (c.y2) {
        int64_t y2_px = 0;
        if (stem || pw.dense || x_scratch || y_post || c.out_int32 || c.res || !y_is_pixel_major(*c.y2, &y2_px)) {
            release_scratch(cache, x_scratch, s);
            release_scratch(cache, y_scratch, s);
            CHX_FAIL(CHX_HIP_EUNSUPPORTED, "QLinearConv pair: needs channels-last x, y1 and y2 and at least 16 input channels");
        }
        a.oc_split = c.oc_split;
        a.y2 = static_cast<char*>(c.y2->data);
        a.y2_px_stride = y2_px;
        a.y2_flip = c.y2_minus_128 ? 0x80808080u : 0u;
        a.q2 = c.rq2.q;
        a.inv_y_scale2 = 1.0f / c.rq2.q.scale;
        a.lo_folded2 = fold_relu_floor(c.rq2.q, c.rq2.relu_floor, c.rne);
    }
    if (stem) {
        ConvStemArgs sa;
        memset(&sa, 0, sizeof(sa));
        const chx_hip_tensor& values = c.x_float ? *c.x_float : x;
        sa.x = static_cast<const char*>(values.data);
        sa.x_n_stride = values.strides[0]; sa.x_c_stride = values.strides[1]; sa.x_h_stride = cs.H > 1 ? values.strides[2] : 0;
        sa.x_float = c.x_float != nullptr;
        sa.xq = c.xq;
        sa.N = cs.N; sa.C = cs.C; sa.H = cs.H; sa.W = cs.W; sa.OH = cs.OH; sa.OW = cs.OW; sa.KH = cs.KH; sa.KW = cs.KW;
        sa.sh = sh; sa.sw = sw; sa.ph = ph; sa.pw = pw_;
        sa.OC = cs.OC;
        sa.wd = pw.wd;
        sa.wsum = pw.wsum;
        sa.x_zp = c.x_zp;
        sa.x_unsigned = x.dtype == CHX_HIP_UINT8 ? 1 : 0;
        sa.corr_mult = sa.x_unsigned ? 128 - c.x_zp : -c.x_zp;
        sa.y = a.y; sa.y_px_stride = a.y_px_stride;
        sa.w_scale = c.w_scale; sa.w_scale_len = c.w_scale_len; sa.bias = c.bias;
        sa.rq = c.rq;
        sa.inv_y_scale = 1.0f / c.rq.q.scale;
        sa.lo_folded = fold_relu_floor(c.rq.q, c.rq.relu_floor, c.rne);
        sa.qp = product_form(c.rq.q, sa.lo_folded, c.rne);
        int rc = launch_conv_stem(sa, c.rne, s);
        if (rc == CHX_HIP_OK && y_post) {
            rc = launch_nhwc_to_nchw_u8(static_cast<const char*>(y_scratch), static_cast<char*>(y.data), cs.N, cs.OC,
                                        (int64_t)cs.OH * cs.OW, (int)a.y_px_stride, s);
        }
        release_scratch(cache, y_scratch, s);
        return rc;
    }
    a.C16 = C16eff;
    {
        // bytes from x to the end of the last pixel's C16 channels (the strides of the three cases above are positive)
        const int64_t n_img = pw.dense ? 1 : cs.N, h_img = pw.dense ? 1 : H, w_img = pw.dense ? (int64_t)cs.N * cs.OH * cs.OW : W;
        const int64_t span = (n_img - 1) * a.x_n_stride + (h_img - 1) * a.x_h_stride + (w_img - 1) * a.x_w_stride + C16eff;
        if (span >= (int64_t(1) << 31) - (int64_t(1) << 24)) {
            release_scratch(cache, x_scratch, s);
            release_scratch(cache, y_scratch, s);
            CHX_FAIL(CHX_HIP_EUNSUPPORTED, "QLinearConv: the activations span 2 GB or more, which the MFMA kernel does not address");
        }
        a.x_bytes = (uint32_t)span;
    }
    a.C64 = pw.C64;
    a.H = H; a.W = W; a.KH = KH; a.KW = KW;
    a.OH = pw.dense ? 1 : cs.OH;
    a.OW = pw.dense ? (int)((int64_t)cs.N * cs.OH * cs.OW) : cs.OW;
    a.sh = sh; a.sw = sw; a.ph = ph; a.pw = pw_;
    a.M = (int64_t)cs.N * cs.OH * cs.OW;
    a.OC = cs.OC;
    a.KP = pw.KP;
    a.bk = pw.BK;
    a.nk = pw.KP / pw.BK;
    a.wp = pw.wp;
    a.wf = pw.wf;
    a.wsum = pw.wsum;
    a.padsum = pw.padsum;
    a.padsum_stride = pw.OCpad;
    a.x_zp = c.x_zp;
    const bool xu = x.dtype == CHX_HIP_UINT8;
    a.corr_mult = xu ? 128 - c.x_zp : -c.x_zp;
    a.w_scale = c.w_scale;
    a.w_scale_len = c.w_scale_len;
    a.bias = c.bias;
    a.rq = c.rq;
    a.inv_y_scale = c.out_int32 ? 0.f : 1.0f / c.rq.q.scale;
    a.lo_folded = fold_relu_floor(c.rq.q, c.rq.relu_floor, c.rne);
    if (!c.out_int32) a.qp = product_form(c.rq.q, a.lo_folded, c.rne);
    if (a.oc_split > 0) {
        a.qp2 = product_form(c.rq2.q, a.lo_folded2, c.rne);
        if ((a.qp.path == 3) != (a.qp2.path == 3)) {  // one form for both
            a.qp = product_form(c.rq.q, a.lo_folded, c.rne, false);
            a.qp2 = product_form(c.rq2.q, a.lo_folded2, c.rne, false);
        }
    }
    if (c.res) a.res = *c.res;
    CHX_REQUIRE(a.M < (int64_t(1) << 31), "QLinearConv: too many output pixels for the MFMA kernel");
    if (c.dq) {
        a.oc_split = kFloatResults;
        a.floats = c.dq;
        a.floats_px_stride = c.dq_px;
        a.floats_zp = c.dq_zpf;
        a.floats_scale = c.dq_scale;
    }
    int toc = 64, tpx = 64, cap = 0, waves = 4;
    pick_tile(c.opt, a, c.out_int32, &toc, &tpx, &cap, &waves);
    if (a.oc_split == kFloatResults) {
        if (!conv_split_takes(a) || (int64_t)((a.OC + 63) / 64) * ((a.M + 63) / 64) > 2048) {
            release_scratch(cache, x_scratch, s);
            CHX_FAIL(CHX_HIP_EUNSUPPORTED, "QLinearConv+DequantizeLinear: not one for the small tiles");
        }
        if (!conv_split_has(toc, tpx, waves)) toc = 32, tpx = 32, cap = 0, waves = 2;
    } else if (a.oc_split % toc != 0) toc = 64, waves = 4, tpx = tpx > 128 ? 128 : tpx;  // (the split is a multiple of 64)
    int rc = CHX_HIP_OK;
    const TunedConfig* tuned = nullptr;
    if (c.tune) {
        for (const TunedConfig& t : c.tune->entries)
            if (t.M == a.M && t.H == a.H && t.W == a.W && t.OH == a.OH && t.OW == a.OW && t.x_n_stride == a.x_n_stride && t.x_h_stride == a.x_h_stride &&
                t.x_w_stride == a.x_w_stride && t.short_form == (a.qp.path != 0) && t.with_res == (c.res != nullptr) && t.oc_split == a.oc_split)
                tuned = &t;
        if (!tuned && c.opt.autotune && !stream_is_capturing(s)) {
            const MeasuredConfigurations::Key key = MeasuredConfigurations::key(a, xu, c.out_int32, c.rne);
            Configuration best;
            if (!measured_configurations().find(key, &best)) {
                rc = tune_conv_mfma(a, xu, c.out_int32, c.rne, s, &best);
                if (rc == CHX_HIP_OK) measured_configurations().add(key, best);
            }
            if (rc == CHX_HIP_OK) {
                c.tune->entries.push_back({a.M, a.H, a.W, a.OH, a.OW, a.x_n_stride, a.x_h_stride, a.x_w_stride, a.qp.path != 0, best.tile_oc, best.tile_px, best.max_wgs_per_cu, best.waves, c.res != nullptr, a.oc_split});
                tuned = &c.tune->entries.back();
            }
        }
    }
    if (tuned) {
        toc = tuned->tile_oc;
        tpx = tuned->tile_px;
        cap = tuned->max_wgs_per_cu;
        waves = tuned->waves;
    }
    if (rc == CHX_HIP_OK) rc = launch_conv_mfma(a, toc, tpx, cap, waves, xu, c.out_int32, c.rne, s);
    if (rc == CHX_HIP_OK && y_post) {
        rc = launch_nhwc_to_nchw_u8(static_cast<const char*>(y_scratch), static_cast<char*>(y.data), cs.N, cs.OC,
                                    (int64_t)cs.OH * cs.OW, (int)a.y_px_stride, s);
    }
    release_scratch(cache, x_scratch, s);
    release_scratch(cache, y_scratch, s);
    return rc;
}

// Reads a small parameter vector back to the host (synchronizes the stream).
int read_back(const chx_hip_tensor& t, std::vector<uint8_t>* out, hipStream_t s) {
    const int64_t n = numel(t);
    out->resize((size_t)n);
    if (n == 0) return CHX_HIP_OK;
    if (t.ndim == 0 || t.strides[0] == 1 || n == 1) {
        CHX_HIP_CALL(hipMemcpyAsync(out->data(), t.data, (size_t)n, hipMemcpyDeviceToHost, s));
    } else {
        CHX_HIP_CALL(hipMemcpy2DAsync(out->data(), 1, t.data, (size_t)t.strides[0], 1, (size_t)n, hipMemcpyDeviceToHost, s));
    }
    CHX_HIP_CALL(hipStreamSynchronize(s));
    return CHX_HIP_OK;
}

bool all_zero(const std::vector<uint8_t>& v) {
    for (uint8_t b : v)
        if (b) return false;
    return true;
}

}  // namespace
}  // namespace chx

using namespace chx;


namespace chx {
namespace {

// Allocates and fills packed weights.  With `persistent` the buffers come from hipMalloc and
// live until release_packed(); otherwise they are stream-ordered scratch.
int make_packed(const chx_hip_tensor& w, bool persistent, hipStream_t s, PackedWeights* pw) {
    const size_t mfma_bytes = packed_bytes((int)w.shape[0], (int)w.shape[1], (int)w.shape[2], (int)w.shape[3], pw);
    const bool stem = pw->dense && stem_shape_fits((int)w.shape[1], (int)w.shape[2], (int)w.shape[3]);
    const size_t stem_bytes =
            stem ? (size_t)(pw->OCpad / 64) * stem_k_blocks((int)w.shape[1], (int)w.shape[2], (int)w.shape[3]) * 2048 : 0;
    // (a call's own weights are read once: not worth another pass; the small tiles take up to 32 taps)
    const size_t fragment_bytes = persistent && (pw->dense || w.shape[2] * w.shape[3] <= 32) ? mfma_bytes : 0;
    // the per-channel sums, and behind them the sixteen classes of border sums
    // (between 2 and 32 taps: the kernel's tap masks hold 32, and a single tap that can lie outside is rare enough for
    // the flat-address padding)
    const bool border_sums = !pw->dense && w.shape[2] * w.shape[3] <= 32 && w.shape[2] * w.shape[3] > 1;
    const size_t sums_bytes = sizeof(int32_t) * pw->OCpad * (border_sums ? 17 : 1), others = mfma_bytes + stem_bytes + sums_bytes;
    // An allocation above 2 MB takes the device runtime 20 us more than one below, and two small ones 1 us more than one: 512 ->
    // 2048 channels in one 57 us for the plan, apart 37.
    const bool apart = fragment_bytes > 0 && others + fragment_bytes > (size_t(2) << 20) && others <= (size_t(2) << 20);
    void* p = nullptr;
    void* p_apart = nullptr;
    if (!persistent) CHX_PROPAGATE(scratch_alloc(&p, others, s));
    else if (spare_memory(&p, others + (apart ? 0 : fragment_bytes), "weights of a convolution") != CHX_HIP_OK) return CHX_HIP_ERUNTIME;
    if (apart && spare_memory(&p_apart, fragment_bytes, "weights of a convolution") != CHX_HIP_OK) {
        (void)hipFree(p);
        return CHX_HIP_ERUNTIME;
    }
    // (weights, and what is made of them, are multiples of 2048 bytes)
    pw->wp = static_cast<int8_t*>(p);
    pw->wd = stem ? pw->wp + mfma_bytes : nullptr;
    pw->wf_apart = static_cast<int8_t*>(p_apart);
    pw->wf = apart ? pw->wf_apart : fragment_bytes ? pw->wp + mfma_bytes + stem_bytes : nullptr;
    pw->wsum = reinterpret_cast<int32_t*>(pw->wp + mfma_bytes + stem_bytes + (apart ? 0 : fragment_bytes));
    pw->padsum = border_sums ? pw->wsum + pw->OCpad : nullptr;
    if (stem) CHX_PROPAGATE(pack_weights_stem(w, pw->OCpad, pw->wd, s));
    if (pw->dense) return pack_weights_dense(w, pw->KP, pw->BK, pw->OCpad, pw->wp, pw->wf, pw->wsum, s);
    return pack_weights(w, pw->C64, pw->BK, pw->OCpad, pw->wp, pw->wf, pw->wsum, pw->padsum, s);
}

void release_packed(PackedWeights* pw, bool persistent, hipStream_t s) {
    if (!persistent) scratch_free(pw->wp, s);
    else if (pw->wp) (void)hipFree(pw->wp);
    if (pw->wf_apart) (void)hipFree(pw->wf_apart);
    pw->wp = pw->wf = pw->wf_apart = pw->wd = nullptr;
    pw->wsum = pw->padsum = nullptr;
}

// Depthwise 3x3 on int8 weights with zero weight zero points: packed filter rows and per-channel sums.
struct DepthwiseState {
    int C = 0;
    void* block = nullptr;  // one allocation: rows | wsum
    int32_t* rows = nullptr;
    int32_t* wsum = nullptr;
};

bool weights_fit_depthwise(const chx_hip_tensor& w, int group) {
    return w.dtype == CHX_HIP_INT8 && group > 1 && w.shape[0] == group && w.shape[1] == 1 && w.shape[2] == 3 &&
           w.shape[3] == 3 && group % 16 == 0;
}

int make_depthwise(const chx_hip_tensor& w, bool persistent, hipStream_t s, DepthwiseState* st) {
    const int C = (int)w.shape[0];
    const size_t rows_bytes = (size_t)(C / 4) * 12 * sizeof(int32_t);
    const size_t total = rows_bytes + (size_t)C * 4;
    void* p = nullptr;
    if (persistent) CHX_HIP_CALL(hipMalloc(&p, total));
    else CHX_PROPAGATE(scratch_alloc(&p, total, s));
    st->C = C;
    st->block = p;
    char* b = static_cast<char*>(p);
    st->rows = reinterpret_cast<int32_t*>(b);
    st->wsum = reinterpret_cast<int32_t*>(b + rows_bytes);
    return pack_depthwise(w, st->rows, st->wsum, s);
}

void release_depthwise(DepthwiseState* st, bool persistent, hipStream_t s) {
    if (!st->block) return;
    if (persistent) (void)hipFree(st->block);
    else scratch_free(st->block, s);
    st->block = nullptr;
}

// channels-last 8-bit tensor whose pixels are 16-byte aligned vectors of C bytes
bool is_depthwise_layout(const chx_hip_tensor& t) {
    if (!is_q8(t.dtype) || t.strides[1] != 1 || !aligned(t.data, 16)) return false;
    for (int ax : {0, 2, 3})
        if (t.shape[ax] != 1 && (t.strides[ax] % 16 != 0 || t.strides[ax] < t.shape[1])) return false;
    return true;
}

struct QConvChecked {
    ConvShape cs;
    ConvDirectArgs direct;
};

// Validation shared by the one-shot call and the plan: everything QLinearConvOp::RunImpl CHECKs.
int check_qconv(
        const chx_hip_tensor* x, float x_scale, int32_t x_zero_point, const chx_hip_tensor* w,
        const chx_hip_tensor* w_scale, const chx_hip_tensor* w_zero_point, float y_scale, int32_t y_zero_point,
        const chx_hip_tensor* bias, const chx_hip_conv_params* params, uint32_t flags, chx_hip_tensor* y, QConvChecked* out) {
    CHX_PROPAGATE(check_tensor(x, "QLinearConv x"));
    CHX_PROPAGATE(check_tensor(w, "QLinearConv w"));
    CHX_PROPAGATE(check_tensor(w_scale, "QLinearConv w_scale"));
    CHX_PROPAGATE(check_tensor(w_zero_point, "QLinearConv w_zero_point"));
    CHX_PROPAGATE(check_tensor(y, "QLinearConv y"));
    CHX_REQUIRE(params != nullptr, "QLinearConv: null params");
    ConvShape& cs = out->cs;
    CHX_PROPAGATE(conv_shape(*x, *w, *params, *y, "QLinearConv", &cs));
    CHX_REQUIRE(w_scale->dtype == CHX_HIP_FLOAT32, "QLinearConv: w_scale must be float32");
    CHX_REQUIRE(w_zero_point->dtype == w->dtype, "QLinearConv: w_zero_point must have the dtype of w");
    // CHECK_EQ(w_scale.GetTotalSize(), w_zero_point.GetTotalSize()), runtime/ops/quantize.cc:76-77
    int64_t slen, sstride, zlen, zstride;
    CHX_PROPAGATE(param_vector(*w_scale, cs.OC, "QLinearConv w_scale", &slen, &sstride));
    CHX_PROPAGATE(param_vector(*w_zero_point, cs.OC, "QLinearConv w_zero_point", &zlen, &zstride));
    CHX_REQUIRE(slen == zlen && w_scale->ndim == w_zero_point->ndim,
                "QLinearConv: w_scale and w_zero_point must have the same shape");
    CHX_REQUIRE(slen == 1 || sstride == 4, "QLinearConv: w_scale must be contiguous");
    ConvDirectArgs& a = out->direct;
    fill_conv_args(*x, *w, *params, *y, cs, &a);
    a.x_zp = x_zero_point;
    a.w_zp = static_cast<const char*>(w_zero_point->data);
    a.w_zp_len = (int32_t)zlen;
    a.w_zp_stride = zstride;
    a.requant = 1;
    a.w_scale = static_cast<const float*>(w_scale->data);
    a.w_scale_len = (int32_t)slen;
    CHX_PROPAGATE(fill_requant(x_scale, y_scale, y_zero_point, *y, bias, cs.OC, flags, "QLinearConv", &a.rq, &a.bias));
    return CHX_HIP_OK;
}

ConvCall conv_call_from(const QConvChecked& q, const chx_hip_tensor* x, chx_hip_tensor* y, const chx_hip_conv_params* p,
                        bool rne, const LaunchOptions& opt) {
    ConvCall c;
    c.opt = opt;
    c.cache = nullptr;
    c.tune = nullptr;
    c.x = x;
    c.y = y;
    c.p = p;
    c.cs = q.cs;
    c.x_zp = q.direct.x_zp;
    c.out_int32 = false;
    c.rne = rne;
    c.w_scale = q.direct.w_scale;
    c.w_scale_len = q.direct.w_scale_len;
    c.bias = q.direct.bias;
    c.rq = q.direct.rq;
    return c;
}

// Runs a depthwise kernel; EUNSUPPORTED when the operands are neither channels-last nor NCHW.
int run_depthwise(const ConvCall& c, const DepthwiseState& st, hipStream_t s) {
    const chx_hip_tensor& x = *c.x;
    const chx_hip_tensor& y = *c.y;
    const bool channels_last = is_depthwise_layout(x) && is_depthwise_layout(y);
    const bool planar = !channels_last && is_q8(x.dtype) && is_q8(y.dtype) && (x.strides[3] == 1 || x.shape[3] == 1) && (y.strides[3] == 1 || y.shape[3] == 1);
    if (!channels_last && !planar)
        CHX_FAIL(CHX_HIP_EUNSUPPORTED, "depthwise kernel needs channels-last 8-bit operands with 16-byte aligned pixels, or NCHW ones");
    if (channels_last && (x.strides[3] * x.shape[3] >= (int64_t(1) << 31) || y.strides[3] * y.shape[3] >= (int64_t(1) << 31)))
        CHX_FAIL(CHX_HIP_EUNSUPPORTED, "depthwise kernel: an input or output row spans 2 GiB or more");
    const bool xs = x.dtype == CHX_HIP_INT8;
    const int32_t zp_u = xs ? c.x_zp + 128 : c.x_zp;
    DepthwiseArgs a;
    memset(&a, 0, sizeof(a));
    a.x = static_cast<const char*>(x.data);
    a.x_n_stride = x.strides[0];
    a.x_h_stride = x.strides[2];
    a.x_w_stride = x.strides[3];
    a.y = static_cast<char*>(y.data);
    a.y_n_stride = y.strides[0];
    a.y_h_stride = y.strides[2];
    a.y_w_stride = y.strides[3];
    a.x_c_stride = x.strides[1];
    a.y_c_stride = y.strides[1];
    a.N = c.cs.N; a.C = c.cs.C; a.H = c.cs.H; a.W = c.cs.W; a.OH = c.cs.OH; a.OW = c.cs.OW;
    a.sh = c.p->stride_h; a.sw = c.p->stride_w; a.ph = c.p->pad_h_begin; a.pw = c.p->pad_w_begin;
    a.x_signed = xs ? 1 : 0;
    a.x_zp_u = zp_u;
    a.rows = st.rows;
    a.wsum = st.wsum;
    a.w_scale = c.w_scale;
    a.w_scale_len = c.w_scale_len;
    a.x_scale = c.rq.x_scale;
    a.bias = c.rq.bias_mode == kBiasNone ? nullptr : c.bias;
    a.float_bias = c.rq.bias_mode == kBiasReferenceFloat ? 1 : 0;
    a.q = c.rq.q;
    a.inv_y_scale = 1.0f / c.rq.q.scale;
    a.lo_folded = fold_relu_floor(c.rq.q, c.rq.relu_floor, c.rne);
    a.qp = product_form(c.rq.q, a.lo_folded, c.rne);
    a.y_flip = c.y_minus_128 ? 0x80808080u : 0u;  // (c.y is then the uint8 view of the caller's int8 array)
    return planar ? launch_depthwise_planar(a, c.rne, s) : launch_depthwise3x3(a, c.rne, s);
}

}  // namespace
}  // namespace chx

namespace chx {
namespace {

// The residual sums fused behind a convolution so far: each one's parameters, and whether constants were found with which
// its two-multiply-add form is exact (find_affine_residual); kept so that the search runs once per set of parameters, also
// for a caller that alternates between a few of them.  Oldest dropped first.
struct SearchedResidual {
    ResidualAdd key, found;
};
constexpr size_t kMaxSearchedResiduals = 8;

// r: channels-last, r_px bytes from pixel to pixel; out_scale within [2^-60, 2^60]
int residual_of(const chx_hip_tensor& r, int64_t r_px, float y_scale, int32_t y_zero_point, int32_t y_dtype, float r_scale, int32_t r_zero_point,
                float out_scale, int32_t out_zero_point, int32_t out_dtype, bool relu, bool wanted, std::vector<SearchedResidual>* searched, hipStream_t s,
                ResidualAdd* out) {
    ResidualAdd res;
    memset(&res, 0, sizeof(res));
    res.r = static_cast<const char*>(r.data);
    res.r_px_stride = r_px;
    res.r_vec_ok = aligned(r.data, 16) && r_px % 16 == 0 ? 1 : 0;
    res.c_flip = y_dtype == CHX_HIP_INT8 ? 0x80808080u : 0u;
    res.r_flip = r.dtype == CHX_HIP_INT8 ? 0x80808080u : 0u;
    res.c_zpf = (float)(y_zero_point + (y_dtype == CHX_HIP_INT8 ? 128 : 0));
    res.c_scale = y_scale;
    res.r_zpf = (float)(r_zero_point + (r.dtype == CHX_HIP_INT8 ? 128 : 0));
    res.r_scale = r_scale;
    res.relu = relu ? 1 : 0;
    res.out = make_quant_params(out_scale, out_zero_point, out_dtype == CHX_HIP_INT8);
    res.inv_out_scale = 1.0f / out_scale;
    res.big = 0x1p40f * out_scale;
    // |DQ(y) + DQ(r)| <= 511 * (|y_scale| + |r_scale|): when that is far below `big`, limiting is the identity
    const double reach = 511.0 * (fabs((double)y_scale) + fabs((double)r_scale));
    res.guard = (reach == reach && reach < 0.25 * (double)res.big) ? 0 : 1;
    // (r's zero point in the unsigned range: a uint8 r with zero point 0, or the same codes stored minus 128 as int8)
    res.lean = out_dtype == CHX_HIP_UINT8 && res.r_zpf == 0.f && out_zero_point == 0 ? 1 : 0;
    // The cheaper form of the sum, where the search over its constants has shown it exact for these parameters.  The
    // search runs on the first call with new parameters (it synchronizes the stream and allocates, so not while the
    // stream is being captured: such a call computes the sum operation by operation).  CHX_HIP_AFFINE_RESIDUAL=0
    // keeps the operation-by-operation arithmetic everywhere.
    {
        ResidualAdd key;
        memcpy(&key, &res, sizeof(key));  // byte copies: the comparison below is one of bytes, padding included
        key.r = nullptr;
        key.r_px_stride = 0;
        key.r_vec_ok = 0;
        const ResidualAdd* known = nullptr;
        for (const SearchedResidual& e : *searched)
            if (memcmp(&key, &e.key, sizeof(key)) == 0) known = &e.found;
        if (wanted && known) {
            res.affine = known->affine;
            res.kc = known->kc;
            res.kr = known->kr;
            res.k0 = known->k0;
            res.floor_pre = known->floor_pre;
        } else if (wanted && !stream_is_capturing(s)) {
            int32_t* counts = nullptr;
            CHX_HIP_CALL(hipMalloc(reinterpret_cast<void**>(&counts), kAffineCandidates * sizeof(int32_t)));
            ResidualAdd found;
            memcpy(&found, &key, sizeof(found));
            const int rc = find_affine_residual(&found, counts, s);
            (void)hipFree(counts);
            CHX_PROPAGATE(rc);
            if (searched->size() == kMaxSearchedResiduals) searched->erase(searched->begin());
            searched->emplace_back();
            memcpy(&searched->back().key, &key, sizeof(key));
            memcpy(&searched->back().found, &found, sizeof(found));
            res.affine = found.affine;
            res.kc = found.kc;
            res.kr = found.kr;
            res.k0 = found.k0;
            res.floor_pre = found.floor_pre;
        }
    }
    memcpy(out, &res, sizeof(res));
    return CHX_HIP_OK;
}

}  // namespace
}  // namespace chx

struct chx_hip_qconv_plan {
    chx_hip_tensor w, w_scale, w_zero_point, bias;
    bool has_bias;
    chx_hip_conv_params params;
    bool mfma;
    bool depthwise;
    chx::DepthwiseState dw;
    chx::PackedWeights pw;
    chx::ScratchCache scratch;  // makes run() unsafe to call concurrently on one plan
    chx::TuneCache tune;
    std::vector<chx::SearchedResidual> searched;  // residual sums fused behind this convolution (run_add)
    chx::LaunchOptions opt;  // read once, when the plan is created
    // recorded runs (HIP graphs) that hold addresses of this plan's packed weights and scratch memory
    int pins = 0;
    bool destroy_when_unpinned = false;
};

extern "C" int chx_hip_qlinear_conv(
        const chx_hip_tensor* x, float x_scale, int32_t x_zero_point, const chx_hip_tensor* w,
        const chx_hip_tensor* w_scale, const chx_hip_tensor* w_zero_point, float y_scale, int32_t y_zero_point,
        const chx_hip_tensor* bias, const chx_hip_conv_params* params, uint32_t flags, chx_hip_tensor* y, void* stream) {
    QConvChecked q;
    CHX_PROPAGATE(check_qconv(x, x_scale, x_zero_point, w, w_scale, w_zero_point, y_scale, y_zero_point, bias, params,
                              flags, y, &q));
    hipStream_t s = as_stream(stream);
    const bool rne = (flags & CHX_HIP_ROUND_ONNX_RNE) != 0;
    if (weights_fit_mfma(*w, params->group)) {
        std::vector<uint8_t> zp;
        CHX_PROPAGATE(read_back(*w_zero_point, &zp, s));
        if (all_zero(zp)) {
            PackedWeights pw;
            CHX_PROPAGATE(make_packed(*w, false, s, &pw));
            const int rc = run_conv_mfma(conv_call_from(q, x, y, params, rne, read_launch_options()), pw, s);
            release_packed(&pw, false, s);
            if (rc != CHX_HIP_EUNSUPPORTED) return rc;
        }
    }
    if (weights_fit_depthwise(*w, params->group)) {
        std::vector<uint8_t> zp;
        CHX_PROPAGATE(read_back(*w_zero_point, &zp, s));
        if (all_zero(zp)) {
            DepthwiseState st;
            CHX_PROPAGATE(make_depthwise(*w, false, s, &st));
            const int rc = run_depthwise(conv_call_from(q, x, y, params, rne, read_launch_options()), st, s);
            release_depthwise(&st, false, s);
            if (rc != CHX_HIP_EUNSUPPORTED) return rc;
        }
    }
    return launch_conv_direct(q.direct, rne, s);
}

namespace chx {
namespace {

// Rank-generic convolutions (ComplementStride / ComplementPad and GroupedConv are rank-generic in the reference,
// runtime/chainerx_util.cc:180-200,313-340).  One spatial axis is a 2-D convolution over images one pixel high and
// takes every kernel the 2-D entry points have; three spatial axes run on the direct kernel, whose outermost spatial
// axis is described here beside the 4-D views (n, c, h, w) that the 2-D checks and argument blocks are made from.
struct ConvNdViews {
    chx_hip_tensor x, w, y;
    chx_hip_conv_params p;
};

chx_hip_tensor drop_axis(const chx_hip_tensor& t, int axis) {
    chx_hip_tensor r = t;
    r.ndim = t.ndim - 1;
    for (int i = axis; i < r.ndim; ++i) {
        r.shape[i] = t.shape[i + 1];
        r.strides[i] = t.strides[i + 1];
    }
    return r;
}

chx_hip_tensor insert_unit_axis(const chx_hip_tensor& t, int axis) {
    chx_hip_tensor r = t;
    r.ndim = t.ndim + 1;
    for (int i = r.ndim - 1; i > axis; --i) {
        r.shape[i] = t.shape[i - 1];
        r.strides[i] = t.strides[i - 1];
    }
    r.shape[axis] = 1;
    r.strides[axis] = t.shape[axis] * t.strides[axis];  // any value serves an axis of extent 1; this one keeps the view dense
    return r;
}

int conv_nd_views(const chx_hip_tensor* x, const chx_hip_tensor* w, const chx_hip_tensor* y, const chx_hip_conv_nd_params* p, const char* op,
                  ConvNdViews* v) {
    CHX_PROPAGATE(check_tensor(x, op));
    CHX_PROPAGATE(check_tensor(w, op));
    CHX_PROPAGATE(check_tensor(y, op));
    CHX_REQUIRE(p != nullptr, "%s: null params", op);
    CHX_REQUIRE(p->n_spatial >= 1 && p->n_spatial <= 3, "%s: %d spatial axes (1, 2 or 3 are computed)", op, p->n_spatial);
    const int nd = p->n_spatial + 2;
    CHX_REQUIRE(x->ndim == nd && w->ndim == nd && y->ndim == nd, "%s: x, w and y must have %d axes for %d spatial ones", op, nd, p->n_spatial);
    const int lead = 3 - p->n_spatial;  // entries of the 2-D parameter block that stay at their neutral values
    int32_t st[3] = {1, 1, 1}, pb[3] = {0, 0, 0}, pe[3] = {0, 0, 0};
    for (int i = 0; i < p->n_spatial; ++i) {
        st[lead + i] = p->stride[i];
        pb[lead + i] = p->pad_begin[i];
        pe[lead + i] = p->pad_end[i];
    }
    v->p.stride_h = st[1]; v->p.stride_w = st[2];
    v->p.pad_h_begin = pb[1]; v->p.pad_w_begin = pb[2];
    v->p.pad_h_end = pe[1]; v->p.pad_w_end = pe[2];
    v->p.group = p->group;
    if (p->n_spatial == 1) {
        v->x = insert_unit_axis(*x, 2);
        v->w = insert_unit_axis(*w, 2);
        v->y = insert_unit_axis(*y, 2);
    } else if (p->n_spatial == 2) {
        v->x = *x; v->w = *w; v->y = *y;
    } else {
        v->x = drop_axis(*x, 2);
        v->w = drop_axis(*w, 2);
        v->y = drop_axis(*y, 2);
    }
    return CHX_HIP_OK;
}

// the outermost spatial axis of a 3-D convolution into the argument block of the direct kernel
int add_depth_axis(const chx_hip_tensor& x, const chx_hip_tensor& w, const chx_hip_tensor& y, const chx_hip_conv_nd_params& p, const char* op,
                   ConvDirectArgs* a) {
    CHX_REQUIRE(p.stride[0] >= 1 && p.pad_begin[0] >= 0 && p.pad_end[0] >= 0, "%s: strides must be positive and pads non-negative", op);
    CHX_REQUIRE(x.shape[2] <= INT32_MAX && w.shape[2] <= INT32_MAX, "%s: extent too large", op);
    const int64_t ed = x.shape[2] + p.pad_begin[0] + p.pad_end[0] - w.shape[2];
    CHX_REQUIRE(ed >= 0, "%s: kernel deeper than the padded input", op);
    const int64_t od = ed / p.stride[0] + 1;
    CHX_REQUIRE(y.shape[2] == od, "%s: y has depth %lld, expected %lld", op, (long long)y.shape[2], (long long)od);
    a->D = (int32_t)x.shape[2];
    a->KD = (int32_t)w.shape[2];
    a->OD = (int32_t)od;
    a->sd = p.stride[0];
    a->pd = p.pad_begin[0];
    a->xsd = x.strides[2];
    a->wsd = w.strides[2];
    a->ysd = y.strides[2];
    a->total *= od;
    return CHX_HIP_OK;
}

}  // namespace
}  // namespace chx

extern "C" int chx_hip_qlinear_conv_nd(
        const chx_hip_tensor* x, float x_scale, int32_t x_zero_point, const chx_hip_tensor* w, const chx_hip_tensor* w_scale,
        const chx_hip_tensor* w_zero_point, float y_scale, int32_t y_zero_point, const chx_hip_tensor* bias,
        const chx_hip_conv_nd_params* params, uint32_t flags, chx_hip_tensor* y, void* stream) {
    ConvNdViews v;
    CHX_PROPAGATE(conv_nd_views(x, w, y, params, "QLinearConv", &v));
    if (params->n_spatial < 3) {
        const int rc = chx_hip_qlinear_conv(&v.x, x_scale, x_zero_point, &v.w, w_scale, w_zero_point, y_scale, y_zero_point, bias, &v.p, flags, &v.y, stream);
        return rc;
    }
    QConvChecked q;
    CHX_PROPAGATE(check_qconv(&v.x, x_scale, x_zero_point, &v.w, w_scale, w_zero_point, y_scale, y_zero_point, bias, &v.p, flags, &v.y, &q));
    CHX_PROPAGATE(add_depth_axis(*x, *w, *y, *params, "QLinearConv", &q.direct));
    return launch_conv_direct(q.direct, (flags & CHX_HIP_ROUND_ONNX_RNE) != 0, as_stream(stream));
}

extern "C" int chx_hip_conv_integer_nd(
        const chx_hip_tensor* x, const chx_hip_tensor* w, int32_t x_zero_point, const chx_hip_tensor* w_zero_point,
        const chx_hip_conv_nd_params* params, chx_hip_tensor* y, void* stream) {
    ConvNdViews v;
    CHX_PROPAGATE(conv_nd_views(x, w, y, params, "ConvInteger", &v));
    if (params->n_spatial < 3) return chx_hip_conv_integer(&v.x, &v.w, x_zero_point, w_zero_point, &v.p, &v.y, stream);
    CHX_REQUIRE(y->dtype == CHX_HIP_INT32, "ConvInteger: y must be int32, got %s", dtype_name(y->dtype));
    ConvShape cs;
    CHX_PROPAGATE(conv_shape(v.x, v.w, v.p, v.y, "ConvInteger", &cs));
    ConvDirectArgs a;
    fill_conv_args(v.x, v.w, v.p, v.y, cs, &a);
    a.x_zp = x_zero_point;
    if (w_zero_point) {
        CHX_PROPAGATE(check_tensor(w_zero_point, "ConvInteger w_zero_point"));
        CHX_REQUIRE(w_zero_point->dtype == w->dtype, "ConvInteger: w_zero_point must have the dtype of w");
        int64_t len, stride;
        CHX_PROPAGATE(param_vector(*w_zero_point, cs.OC, "ConvInteger w_zero_point", &len, &stride));
        a.w_zp = static_cast<const char*>(w_zero_point->data);
        a.w_zp_len = (int32_t)len;
        a.w_zp_stride = stride;
    }
    CHX_PROPAGATE(add_depth_axis(*x, *w, *y, *params, "ConvInteger", &a));
    return launch_conv_direct(a, false, as_stream(stream));
}

extern "C" int chx_hip_qconv_plan_create(
        const chx_hip_tensor* w, const chx_hip_tensor* w_scale, const chx_hip_tensor* w_zero_point,
        const chx_hip_tensor* bias, const chx_hip_conv_params* params, void* stream, chx_hip_qconv_plan** plan) {
    CHX_REQUIRE(plan != nullptr, "QLinearConv plan: null output");
    *plan = nullptr;
    CHX_PROPAGATE(check_tensor(w, "QLinearConv w"));
    CHX_PROPAGATE(check_tensor(w_scale, "QLinearConv w_scale"));
    CHX_PROPAGATE(check_tensor(w_zero_point, "QLinearConv w_zero_point"));
    CHX_REQUIRE(params != nullptr, "QLinearConv plan: null params");
    CHX_REQUIRE(w->ndim == 4 && is_q8(w->dtype), "QLinearConv plan: w must be a 4-D uint8/int8 tensor");
    if (bias) CHX_PROPAGATE(check_tensor(bias, "QLinearConv bias"));
    hipStream_t s = as_stream(stream);
    chx_hip_qconv_plan* p = new chx_hip_qconv_plan();
    p->w = *w;
    p->w_scale = *w_scale;
    p->w_zero_point = *w_zero_point;
    p->has_bias = bias != nullptr;
    if (bias) p->bias = *bias;
    p->params = *params;
    p->mfma = false;
    p->depthwise = false;
    p->opt = chx::read_launch_options();
    if (weights_fit_depthwise(*w, params->group) && w_zero_point->dtype == w->dtype && w_zero_point->ndim <= 1) {
        std::vector<uint8_t> zp;
        int rc = read_back(*w_zero_point, &zp, s);
        if (rc == CHX_HIP_OK && all_zero(zp)) {
            rc = make_depthwise(*w, true, s, &p->dw);
            if (rc == CHX_HIP_OK && hipStreamSynchronize(s) != hipSuccess) rc = CHX_HIP_ERUNTIME;
            if (rc == CHX_HIP_OK) p->depthwise = true;
        }
        if (rc != CHX_HIP_OK) {
            release_depthwise(&p->dw, true, s);
            delete p;
            return rc;
        }
    }
    if (weights_fit_mfma(*w, params->group) && w_zero_point->dtype == w->dtype && w_zero_point->ndim <= 1) {
        std::vector<uint8_t> zp;
        int rc = read_back(*w_zero_point, &zp, s);
        if (rc == CHX_HIP_OK && all_zero(zp)) {
            rc = make_packed(*w, true, s, &p->pw);
            if (rc == CHX_HIP_OK) {
                hipError_t e = hipStreamSynchronize(s);
                if (e != hipSuccess) {
                    set_error("hipStreamSynchronize failed: %s", hipGetErrorString(e));
                    rc = CHX_HIP_ERUNTIME;
                }
            }
            if (rc == CHX_HIP_OK) p->mfma = true;
        }
        if (rc != CHX_HIP_OK) {
            release_packed(&p->pw, true, s);
            delete p;
            return rc;
        }
    }
    *plan = p;
    return CHX_HIP_OK;
}

namespace chx {
namespace {
// CHX_HIP_STORE_MINUS_128: the array is int8, its quantization is that of the uint8 array it stands for.  *view is what
// the checks and the requantization parameters are derived from.
int result_view(const chx_hip_tensor* y, uint32_t flags, const char* op, chx_hip_tensor* view, bool* minus_128) {
    CHX_PROPAGATE(check_tensor(y, op));
    *view = *y;
    *minus_128 = (flags & CHX_HIP_STORE_MINUS_128) != 0;
    if (*minus_128) {
        CHX_REQUIRE(y->dtype == CHX_HIP_INT8, "%s: codes minus 128 are stored into an int8 array, got %s", op, dtype_name(y->dtype));
        view->dtype = CHX_HIP_UINT8;
    }
    return CHX_HIP_OK;
}
}  // namespace
}  // namespace chx

extern "C" int chx_hip_qconv_plan_run(
        const chx_hip_qconv_plan* plan, const chx_hip_tensor* x, float x_scale, int32_t x_zero_point, float y_scale,
        int32_t y_zero_point, uint32_t flags, chx_hip_tensor* y, void* stream) {
    CHX_REQUIRE(plan != nullptr, "QLinearConv plan: null plan");
    chx_hip_tensor yv;
    bool minus_128 = false;
    CHX_PROPAGATE(result_view(y, flags, "QLinearConv y", &yv, &minus_128));
    QConvChecked q;
    CHX_PROPAGATE(check_qconv(x, x_scale, x_zero_point, &plan->w, &plan->w_scale, &plan->w_zero_point, y_scale,
                              y_zero_point, plan->has_bias ? &plan->bias : nullptr, &plan->params, flags, &yv, &q));
    hipStream_t s = as_stream(stream);
    const bool rne = (flags & CHX_HIP_ROUND_ONNX_RNE) != 0;
    if (plan->mfma) {
        ConvCall call = conv_call_from(q, x, &yv, &plan->params, rne, plan->opt);
        call.cache = const_cast<ScratchCache*>(&plan->scratch);
        call.tune = const_cast<TuneCache*>(&plan->tune);
        call.y_minus_128 = minus_128;
        const int rc = run_conv_mfma(call, plan->pw, s);
        if (rc != CHX_HIP_EUNSUPPORTED || minus_128) return rc;
    }
    if (plan->depthwise) {
        ConvCall call = conv_call_from(q, x, &yv, &plan->params, rne, plan->opt);
        call.y_minus_128 = minus_128;
        const int rc = run_depthwise(call, plan->dw, s);
        if (rc != CHX_HIP_EUNSUPPORTED || minus_128) return rc;
    }
    if (minus_128) CHX_FAIL(CHX_HIP_EUNSUPPORTED, "QLinearConv: codes minus 128 are stored by the matrix-core and the depthwise kernel only");
    return launch_conv_direct(q.direct, rne, s);
}

extern "C" int chx_hip_qconv_plan_run_quantize(
        const chx_hip_qconv_plan* plan, const chx_hip_tensor* x, float q_scale, int32_t q_zero_point, float x_scale, int32_t x_zero_point,
        float y_scale, int32_t y_zero_point, uint32_t flags, chx_hip_tensor* y, void* stream) {
    CHX_REQUIRE(plan != nullptr, "QuantizeLinear+QLinearConv: null plan");
    CHX_PROPAGATE(check_tensor(x, "QuantizeLinear+QLinearConv x"));
    CHX_PROPAGATE(check_tensor(y, "QuantizeLinear+QLinearConv y"));
    CHX_REQUIRE(x->dtype == CHX_HIP_FLOAT32, "QuantizeLinear+QLinearConv: x must be float32, got %s", dtype_name(x->dtype));
    CHX_REQUIRE(q_zero_point >= 0 && q_zero_point <= 255, "QuantizeLinear+QLinearConv: zero point %d outside the range of uint8", q_zero_point);
    if (flags & (CHX_HIP_STORE_MINUS_128 | CHX_HIP_ROUND_ONNX_RNE))
        CHX_FAIL(CHX_HIP_EUNSUPPORTED, "QuantizeLinear+QLinearConv: the reference's rounding and plain codes only");
    // the codes as they would lie, were there an array of them
    chx_hip_tensor codes = *x;
    codes.dtype = CHX_HIP_UINT8;
    for (int i = 0; i < x->ndim; ++i) {
        if (x->strides[i] % 4 != 0) CHX_FAIL(CHX_HIP_EUNSUPPORTED, "QuantizeLinear+QLinearConv: floats at any byte");
        codes.strides[i] /= 4;
    }
    if (reinterpret_cast<uintptr_t>(x->data) % 4 != 0) CHX_FAIL(CHX_HIP_EUNSUPPORTED, "QuantizeLinear+QLinearConv: floats at any byte");
    QConvChecked q;
    CHX_PROPAGATE(check_qconv(&codes, x_scale, x_zero_point, &plan->w, &plan->w_scale, &plan->w_zero_point, y_scale, y_zero_point,
                              plan->has_bias ? &plan->bias : nullptr, &plan->params, flags, y, &q));
    if (byte_ranges_overlap(*y, *x)) CHX_FAIL(CHX_HIP_EUNSUPPORTED, "QuantizeLinear+QLinearConv: x and y overlap in memory");
    const QuantProduct xq = product_form_of_any_value(make_quant_params(q_scale, q_zero_point, false));
    if (!plan->mfma || xq.path == 0) CHX_FAIL(CHX_HIP_EUNSUPPORTED, "QuantizeLinear+QLinearConv: no short form of this quantization, or weights for another kernel");
    ConvCall call = conv_call_from(q, &codes, y, &plan->params, false, plan->opt);
    call.cache = const_cast<ScratchCache*>(&plan->scratch);
    call.tune = const_cast<TuneCache*>(&plan->tune);
    call.x_float = x;
    call.xq = xq;
    return run_conv_mfma(call, plan->pw, as_stream(stream));
}

// CHX_HIP_MOST_DEQUANTIZED: two launches and one inside a recording, us: 8 x 2048 -> 1000 7.3 and 5.3, 128 x 1280
// -> 1000 8.5 and 5.9, 512 x 2048 -> 1000 14.8 and 8.5, 100 x 4096 -> 4096 15.1 and 12.8; beyond, the small tiles read their operands too often:
// 4 x 2048 -> 256 at 32x32 (a million results) 12.4 and 16.0, 8 x 1024 -> 512 at 28x28 14.2 and 24.3.
extern "C" int chx_hip_qconv_plan_run_dequantize(
        const chx_hip_qconv_plan* plan, const chx_hip_tensor* x, float x_scale, int32_t x_zero_point, float y_scale, int32_t y_zero_point, int32_t y_dtype,
        uint32_t flags, float dq_scale, int32_t dq_zero_point, chx_hip_tensor* y, void* stream) {
    CHX_REQUIRE(plan != nullptr, "QLinearConv+DequantizeLinear: null plan");
    CHX_PROPAGATE(check_tensor(x, "QLinearConv+DequantizeLinear x"));
    CHX_PROPAGATE(check_tensor(y, "QLinearConv+DequantizeLinear y"));
    CHX_REQUIRE(y->dtype == CHX_HIP_FLOAT32, "QLinearConv+DequantizeLinear: y must be float32, got %s", dtype_name(y->dtype));
    CHX_REQUIRE(is_q8(y_dtype), "QLinearConv+DequantizeLinear: the codes must be uint8 or int8");
    if (flags & CHX_HIP_STORE_MINUS_128) CHX_FAIL(CHX_HIP_EUNSUPPORTED, "QLinearConv+DequantizeLinear: plain codes only");
    // the codes as they would lie, were there an array of them
    chx_hip_tensor codes = *y;
    codes.dtype = y_dtype;
    bool whole = reinterpret_cast<uintptr_t>(y->data) % 4 == 0;
    for (int i = 0; i < y->ndim; ++i) {
        whole = whole && y->strides[i] % 4 == 0;
        codes.strides[i] /= 4;
    }
    QConvChecked q;
    CHX_PROPAGATE(check_qconv(x, x_scale, x_zero_point, &plan->w, &plan->w_scale, &plan->w_zero_point, y_scale, y_zero_point,
                              plan->has_bias ? &plan->bias : nullptr, &plan->params, flags, &codes, &q));
    int64_t px = 0;
    if (!plan->mfma || !whole || !y_is_pixel_major(codes, &px) || plan->w.shape[2] != 1 || plan->w.shape[3] != 1 || numel(codes) > CHX_HIP_MOST_DEQUANTIZED || byte_ranges_overlap(*y, *x) ||
        (plan->opt.forced_tile && !conv_split_has(plan->opt.tile_oc, plan->opt.tile_px, plan->opt.waves)))
        CHX_FAIL(CHX_HIP_EUNSUPPORTED, "QLinearConv+DequantizeLinear: 1x1 filters, few channels-last results that do not overlap x");
    ConvCall call = conv_call_from(q, x, &codes, &plan->params, (flags & CHX_HIP_ROUND_ONNX_RNE) != 0, plan->opt);
    call.cache = const_cast<ScratchCache*>(&plan->scratch);
    call.tune = const_cast<TuneCache*>(&plan->tune);
    call.dq = static_cast<float*>(y->data);
    call.dq_px = px;
    call.dq_zpf = (float)dq_zero_point;
    call.dq_scale = dq_scale;
    return run_conv_mfma(call, plan->pw, as_stream(stream));
}

extern "C" int chx_hip_qconv_plan_run_pair(
        const chx_hip_qconv_plan* plan, const chx_hip_tensor* x, float x_scale, int32_t x_zero_point, int32_t split,
        float y1_scale, int32_t y1_zero_point, uint32_t flags1, chx_hip_tensor* y1, float y2_scale, int32_t y2_zero_point,
        uint32_t flags2, chx_hip_tensor* y2, void* stream) {
    CHX_REQUIRE(plan != nullptr, "QLinearConv pair: null plan");
    chx_hip_tensor y1v, y2v;
    bool y1_minus_128 = false, y2_minus_128 = false;
    CHX_PROPAGATE(result_view(y1, flags1, "QLinearConv pair y1", &y1v, &y1_minus_128));
    CHX_PROPAGATE(result_view(y2, flags2, "QLinearConv pair y2", &y2v, &y2_minus_128));
    CHX_REQUIRE(y1->ndim == 4 && y2->ndim == 4, "QLinearConv pair: y1 and y2 must be 4-D");
    const int64_t OC = plan->w.shape[0];
    CHX_REQUIRE(split > 0 && split < OC && y1->shape[1] == split && y2->shape[1] == OC - split,
                "QLinearConv pair: y1 and y2 must hold the first %d and the other %lld of the plan's %lld output channels", split,
                (long long)(OC - split), (long long)OC);
    for (int ax : {0, 2, 3}) CHX_REQUIRE(y1->shape[ax] == y2->shape[ax], "QLinearConv pair: y1 and y2 differ in batch or image size");
    const uint32_t shared = CHX_HIP_BIAS_ONNX_INT32 | CHX_HIP_ROUND_ONNX_RNE;
    CHX_REQUIRE((flags1 & shared) == (flags2 & shared), "QLinearConv pair: the two halves must agree on the bias and rounding flags");
    CHX_PROPAGATE(check_tensor(x, "QLinearConv pair x"));
    CHX_REQUIRE(!byte_ranges_overlap(*y1, *x) && !byte_ranges_overlap(*y2, *x) && !byte_ranges_overlap(*y1, *y2),
                "QLinearConv pair: x, y1 and y2 must not overlap in memory");
    if (split % 64 != 0) CHX_FAIL(CHX_HIP_EUNSUPPORTED, "QLinearConv pair: the first convolution must have a multiple of 64 output channels");
    if (!plan->mfma) CHX_FAIL(CHX_HIP_EUNSUPPORTED, "QLinearConv pair: these weights do not run on the matrix-core kernel");
    // shapes and parameters as for one convolution with all output channels, laid out like y1
    chx_hip_tensor y_all = y1v;
    y_all.shape[1] = OC;
    QConvChecked q;
    CHX_PROPAGATE(check_qconv(x, x_scale, x_zero_point, &plan->w, &plan->w_scale, &plan->w_zero_point, y1_scale, y1_zero_point,
                              plan->has_bias ? &plan->bias : nullptr, &plan->params, flags1, &y_all, &q));
    RequantParams rq2;
    const int32_t* bias2 = nullptr;
    CHX_PROPAGATE(fill_requant(x_scale, y2_scale, y2_zero_point, y2v, plan->has_bias ? &plan->bias : nullptr, OC, flags2,
                               "QLinearConv pair", &rq2, &bias2));
    hipStream_t s = as_stream(stream);
    ConvCall call = conv_call_from(q, x, &y1v, &plan->params, (flags1 & CHX_HIP_ROUND_ONNX_RNE) != 0, plan->opt);
    call.cache = const_cast<ScratchCache*>(&plan->scratch);
    call.tune = const_cast<TuneCache*>(&plan->tune);
    call.y2 = &y2v;
    call.y_minus_128 = y1_minus_128;
    call.y2_minus_128 = y2_minus_128;
    call.oc_split = split;
    call.rq2 = rq2;
    return run_conv_mfma(call, plan->pw, s);
}

extern "C" int chx_hip_qconv_plan_run_add(
        const chx_hip_qconv_plan* plan, const chx_hip_tensor* x, float x_scale, int32_t x_zero_point, float y_scale,
        int32_t y_zero_point, int32_t y_dtype, uint32_t flags, const chx_hip_tensor* r, float r_scale, int32_t r_zero_point,
        float out_scale, int32_t out_zero_point, int32_t relu, chx_hip_tensor* out, void* stream) {
    CHX_REQUIRE(plan != nullptr, "QLinearConv+Add: null plan");
    CHX_PROPAGATE(check_tensor(r, "QLinearConv+Add r"));
    // (with CHX_HIP_STORE_MINUS_128 `out` is an int8 array that holds the codes of a uint8 sum minus 128)
    chx_hip_tensor outv;
    bool out_minus_128 = false;
    CHX_PROPAGATE(result_view(out, flags, "QLinearConv+Add out", &outv, &out_minus_128));
    const int32_t out_dtype = outv.dtype;
    CHX_REQUIRE(is_q8(y_dtype) && is_q8(r->dtype) && is_q8(out_dtype), "QLinearConv+Add: y, r and out must be uint8 or int8");
    CHX_REQUIRE(r->ndim == 4 && out->ndim == 4, "QLinearConv+Add: r and out must be 4-D");
    for (int i = 0; i < 4; ++i)
        CHX_REQUIRE(r->shape[i] == out->shape[i], "QLinearConv+Add: r and out differ in shape (no broadcasting)");
    auto in_range = [](int32_t zp, int32_t dt) { return dt == CHX_HIP_INT8 ? zp >= -128 && zp <= 127 : zp >= 0 && zp <= 255; };
    CHX_REQUIRE(in_range(r_zero_point, r->dtype) && in_range(out_zero_point, out_dtype),
                "QLinearConv+Add: zero point out of the range of its type");
    if (!(out_scale >= 0x1p-60f && out_scale <= 0x1p60f))
        CHX_FAIL(CHX_HIP_EUNSUPPORTED, "QLinearConv+Add: out_scale outside [2^-60, 2^60]");
    // `out` is written while x and r are still being read (and, when the launch configurations are timed,
    // several times over)
    CHX_PROPAGATE(check_tensor(x, "QLinearConv+Add x"));
    CHX_REQUIRE(!byte_ranges_overlap(*out, *x) && !byte_ranges_overlap(*out, *r), "QLinearConv+Add: out overlaps x or r in memory");
    // the convolution's own result has the layout of `out` and the type y_dtype
    chx_hip_tensor y = *out;
    y.dtype = y_dtype;
    QConvChecked q;
    CHX_PROPAGATE(check_qconv(x, x_scale, x_zero_point, &plan->w, &plan->w_scale, &plan->w_zero_point, y_scale,
                              y_zero_point, plan->has_bias ? &plan->bias : nullptr, &plan->params, flags, &y, &q));
    if (!plan->mfma) CHX_FAIL(CHX_HIP_EUNSUPPORTED, "QLinearConv+Add: these weights do not run on the matrix-core kernel");
    int64_t r_px = 0, o_px = 0;
    if (!y_is_pixel_major(*r, &r_px) || !y_is_pixel_major(*out, &o_px))
        CHX_FAIL(CHX_HIP_EUNSUPPORTED, "QLinearConv+Add: r and out must be channels-last");
    ResidualAdd res;
    hipStream_t s = as_stream(stream);
    CHX_PROPAGATE(residual_of(*r, r_px, y_scale, y_zero_point, y_dtype, r_scale, r_zero_point, out_scale, out_zero_point, out_dtype, relu != 0,
                              plan->opt.affine_residual, &const_cast<chx_hip_qconv_plan*>(plan)->searched, s, &res));
    ConvCall call = conv_call_from(q, x, &y, &plan->params, (flags & CHX_HIP_ROUND_ONNX_RNE) != 0, plan->opt);
    call.cache = const_cast<ScratchCache*>(&plan->scratch);
    call.tune = const_cast<TuneCache*>(&plan->tune);
    call.res = &res;
    call.y_minus_128 = out_minus_128;
    return run_conv_mfma(call, plan->pw, s);
}

extern "C" int chx_hip_qconv_plan_describe(const chx_hip_qconv_plan* plan, char* buf, size_t buf_size) {
    CHX_REQUIRE(plan != nullptr && buf != nullptr && buf_size > 0, "QLinearConv plan: null argument");
    std::string text;
    for (const TunedConfig& t : plan->tune.entries) {
        const bool lds = t.max_wgs_per_cu == kConvSame || (t.max_wgs_per_cu == kConvSplitPatch && conv_split_has(t.tile_oc, t.tile_px, t.waves));
        char line[160];
        snprintf(line, sizeof(line), "M=%lld %dx%d res=%d tile=%dx%d wgs_per_cu=%d waves=%d%s\n", (long long)t.M, t.OH, t.OW, t.with_res ? 1 : 0,
                 t.tile_oc, t.tile_px, lds ? 0 : t.max_wgs_per_cu, t.waves, lds ? " pixels=lds" : "");
        text += line;
    }
    if (!plan->searched.empty()) text += plan->searched.back().found.affine ? "residual=affine\n" : "residual=exact\n";
    strncpy(buf, text.c_str(), buf_size - 1);
    buf[buf_size - 1] = 0;
    return CHX_HIP_OK;
}

extern "C" int chx_hip_qconv_plan_pin(chx_hip_qconv_plan* plan, int32_t delta) {
    CHX_REQUIRE(plan != nullptr && (delta == 1 || delta == -1), "QLinearConv plan pin: a plan and +1 or -1");
    CHX_REQUIRE(plan->pins + delta >= 0, "QLinearConv plan pin: released more often than pinned");
    plan->pins += delta;
    plan->scratch.pinned = plan->pins > 0;
    if (plan->pins == 0 && plan->destroy_when_unpinned) {
        plan->destroy_when_unpinned = false;
        chx_hip_qconv_plan_destroy(plan);
    }
    return CHX_HIP_OK;
}

extern "C" void chx_hip_qconv_plan_destroy(chx_hip_qconv_plan* plan) {
    if (!plan) return;
    if (plan->pins > 0) {
        // a recorded run still launches kernels on this plan's memory: it goes when the last pin does
        plan->destroy_when_unpinned = true;
        return;
    }
    chx::release_packed(&plan->pw, true, nullptr);
    chx::release_depthwise(&plan->dw, true, nullptr);
    for (int i = 0; i < 2; ++i)
        if (plan->scratch.ptr[i]) (void)hipFree(plan->scratch.ptr[i]);
    delete plan;
}

namespace chx {
namespace {
double padded(int64_t n, int64_t by) {
    return (double)((n + by - 1) / by * by);
}

// Whether a ConvInteger with 1x1 filters that could be a product is one of those for which another kernel is faster, as far as
// that kernel takes it.
//  * Planar: a product is padded to tiles of 128 columns of an image and of 32 filters, and where rows do not start at lines of 128 bytes two tiles
//    write parts of one.  Both times in us, fitted to 346 calls of 16 to 2048 channels in, 8 to 2048 out and images of 4 to 80, measured both ways (within
//    20 and 15 %).  All as products were 0.67 of the others' time on average and 46 slower by more than 5 % (up to 3.1 times: 73 x 1640 -> 960 at 5x5 26
//    and 80); by this choice 0.65, six of them, by up to 10 % (of 600 others, planar and not, one, 70 x 672 -> 72 at 5x5: 10.3 and 14.0).
//  * Channels-last with strides, fewer filters than 0.3 of the channels and one launch (conv_strip.hip), in us there and as a product: 21 x 176 -> 16 at 34x34 8.7 and
//    11.5, 55 x 672 -> 80 at 5x5 11.2 and 19.2; more filters (10 x 136 -> 320 at 24x24, 11.6 and 8.4) gain by the product, by 14 % on average.
//  * Channels-last with strides and rows of no more than half a tile of 16, by what the two kernels' work comes to: 64 x 1024 -> 2048
//    at 7x7 84 and 130, 62 x 544 -> 1312 at 4x4 22.1 and 32.6; 135 x 552 -> 304 at 7x7 61.3 and 27.6.
bool faster_than_product(const chx_hip_conv_params& p, const ConvShape& cs, const ConvDirectArgs& a, bool channels_last) {
    const int64_t C = a.C, OC = cs.OC, columns = (int64_t)cs.OH * cs.OW;
    if (!channels_last) {
        const double N = cs.N, pixels = N * columns, filters = padded(OC, 32), channels = padded(C, 32), results = 4e-6 * (double)a.total;
        const double product = 4.7 + N * padded(columns, 128) * filters * (3.41e-9 * channels + 0.165e-6) + (columns % 32 == 0 ? 0.044 : 0.121) * results;
        const double other = 6.9 + pixels * (0.737e-9 * filters * channels + 0.432e-6 * C) + 0.126 * results + 0.541e-6 * N * C * padded(columns, 64) + 2.7e-6 * OC * C +
                             0.313e-6 * N * ((cs.OW + 3) / 4) * cs.OH * filters * ((C + 31) / 32);
        return product > 0.88 * other;
    }
    if ((p.stride_h == 1 && p.stride_w == 1) || p.stride_h != p.stride_w || p.stride_h > 2) return false;
    if (conv_strip_takes(a)) return 10 * OC <= 3 * C;
    if (cs.OW > 8) return false;
    const double steps = (double)cs.N * cs.OH * ((OC + 63) / 64) * ((C + 63) / 64);
    const double planes = 12.0 + 2.5e-6 * (double)cs.N * (double)C * (double)cs.H * (double)cs.W + 4e-9 * (double)a.total * (double)C + 2e-6 * (double)a.total;
    return planes < 0.9 * (7.0 + 0.45e-3 * steps);
}

// Whether a channels-last ConvInteger with 1x1 filters that the packed kernel takes is faster there.  That reads the filters' zero points back and packs
// them, 73 us whatever the size; a product needs none of it, but its kernel is the slower one, and its tiles are of 128 filters.  Both times in us, fitted to 182
// calls of 5 to 30 G multiply-adds, measured both ways (within 8 and 15 %): by this choice 0.95 of the packed kernel's time on average, none slower
// by more than 6 % (of 350 others one, by 11 %).  64 x 512 -> 512 channels at 56x56 221 packed and 276 as a product, 64 x 1024 -> 1024 at 28x28 164 and 250; 20 x 512 -> 280 at 72x72 81
// and 111, with few filters beside a tile; 256 -> 384 channels at 39 G 208 and 166.  With few pixels to a filter its packing is what counts (64 images of 7x7, 2048 -> 3072: 145
// and 101), and with strides the product's tiles are rows of results (138 x 2000 -> 376 at 11x11, 12.6 G: 75 and 162; of 40 such calls from 8 G on, 13 slower, by up to 4.3 times).
bool faster_packed(const chx_hip_conv_params& p, const ConvShape& cs, const ConvDirectArgs& a) {
    if (p.stride_h != 1 || p.stride_w != 1) return true;
    const int64_t pixels = (int64_t)cs.N * cs.OH * cs.OW;
    if (pixels < 8192) return false;
    const double results = 4e-6 * (double)a.total;
    const double product = 7.6 + 4.37e-9 * (double)pixels * padded(cs.OC, 128) * padded(a.C, 32) + 0.069 * results;
    const double packed = 8.7 + (double)pixels * (1.7e-9 * padded(cs.OC, 64) * padded(a.C, 64) + 0.155e-6 * a.C + 17.5e-6) + 0.305 * results;
    return product > 0.95 * std::max(73.0, packed);
}

// A ConvInteger with 1x1 filters as the product that it is, on gemm_i8.hip: pixels by filters where x and y are channels-last and
// dense (with strides above 1 a product for every row of results), filters by pixels for every image where both are planar (one zero point for all filters: there it is that of the
// rows).  EUNSUPPORTED, with nothing launched, for anything else and, unless `any`, for what faster_than_product() names.  The other kernels bring channels-last pixels into planes
// first and keep strips of few filters; us there and here: 5 x 80 -> 24 channels at 11x11, channels-last 9.0 and 6.2, 36 x 96 -> 56 at
// 32x32 17.2 and 7.5; planar 37 x 48 -> 224 at 16x16 11.4 and 6.4, 56 x 168 -> 32 at 39x39 28.9 and 9.3, with few of both the same (3 x
// 48 -> 24 at 55x55 6.3 and 6.3).  Stride 2, channels-last: 9 x 48 -> 40 at 8x8 8.8 and 6.3, 40 x 40 -> 152 at 24x24 9.7 and 6.4.
int run_conv_as_product(const chx_hip_tensor& x, const chx_hip_tensor& w, int32_t x_zero_point, const chx_hip_conv_params& p, const ConvShape& cs, const ConvDirectArgs& a, const chx_hip_tensor& y, bool any, hipStream_t s) {
    // (pads at the ends with stride 1 would show in OH and OW; with larger strides the last window has to lie inside)
    if (cs.KH != 1 || cs.KW != 1 || p.group != 1 || p.pad_h_begin != 0 || p.pad_w_begin != 0 || (cs.OH - 1) * p.stride_h >= cs.H || (cs.OW - 1) * p.stride_w >= cs.W) return CHX_HIP_EUNSUPPORTED;
    const bool dense = p.stride_h == 1 && p.stride_w == 1;
    const int64_t C = x.shape[1], OC = cs.OC, HW = (int64_t)cs.OH * cs.OW;
    if ((C != 1 && w.strides[1] != 1) || a.total == 0) return CHX_HIP_EUNSUPPORTED;
    MatMulDirectArgs m;
    memset(&m, 0, sizeof(m));
    int64_t x_px = 0, y_px = 0;
    m.y = static_cast<char*>(y.data);
    m.total = a.total;
    m.K = C;
    m.lds_64k = 1;  // (a ConvInteger asks for no more than any launch may: the split kernel only)
    if (y_is_pixel_major(x, &x_px) && y_is_pixel_major(y, &y_px)) {
        if (!any && faster_than_product(p, cs, a, true)) return CHX_HIP_EUNSUPPORTED;
        m.a = static_cast<const char*>(x.data);
        m.b = static_cast<const char*>(w.data);
        m.M = cs.N * HW;
        m.N = OC;
        m.a_row = x_px; m.a_col = 1;
        if (!dense) {  // a product for every row of results, whose first pixels have to be equally far apart
            if (cs.N > 1 && cs.H != cs.OH * p.stride_h) return CHX_HIP_EUNSUPPORTED;
            m.M = cs.OW;
            m.a_row = p.stride_w * x_px;
            m.a_batch = (int64_t)p.stride_h * cs.W * x_px;
            m.y_batch = cs.OW * y_px;
        }
        m.b_row = 1; m.b_col = w.strides[0];
        m.y_row = y_px; m.y_col = 4;
        m.a_signed = x.dtype == CHX_HIP_INT8;
        m.b_signed = w.dtype == CHX_HIP_INT8;
        m.a_zp_imm = x_zero_point;
        m.b_zp = a.w_zp;
        m.b_zp_len = a.w_zp_len;
        m.b_zp_stride = a.w_zp_stride;
        m.b_zp_signed = m.b_signed;
        return launch_matmul_i8(m, false, s);
    }
    const bool planar = dense && (cs.OW == 1 || (x.strides[3] == 1 && y.strides[3] == 4)) && (cs.OH == 1 || (x.strides[2] == x.shape[3] && y.strides[2] == 4 * x.shape[3]));
    if (planar && a.w_zp_len <= 1) {
        if (!any && faster_than_product(p, cs, a, false)) return CHX_HIP_EUNSUPPORTED;
        m.a = static_cast<const char*>(w.data);
        m.b = static_cast<const char*>(x.data);
        m.M = OC;
        m.N = HW;
        m.a_row = w.strides[0]; m.a_col = 1;
        m.b_batch = x.strides[0]; m.b_row = x.strides[1]; m.b_col = 1;
        m.y_batch = y.strides[0]; m.y_row = y.strides[1]; m.y_col = 4;
        m.a_signed = w.dtype == CHX_HIP_INT8;
        m.b_signed = x.dtype == CHX_HIP_INT8;
        m.a_zp = a.w_zp;
        m.a_zp_len = a.w_zp_len;
        m.a_zp_signed = m.a_signed;
        m.b_zp_imm = x_zero_point;
        return launch_matmul_i8(m, false, s);
    }
    return CHX_HIP_EUNSUPPORTED;
}
}  // namespace
}  // namespace chx

extern "C" int chx_hip_conv_integer(
        const chx_hip_tensor* x, const chx_hip_tensor* w, int32_t x_zero_point, const chx_hip_tensor* w_zero_point,
        const chx_hip_conv_params* params, chx_hip_tensor* y, void* stream) {
    CHX_PROPAGATE(check_tensor(x, "ConvInteger x"));
    CHX_PROPAGATE(check_tensor(w, "ConvInteger w"));
    CHX_PROPAGATE(check_tensor(y, "ConvInteger y"));
    CHX_REQUIRE(params != nullptr, "ConvInteger: null params");
    CHX_REQUIRE(y->dtype == CHX_HIP_INT32, "ConvInteger: y must be int32, got %s", dtype_name(y->dtype));
    ConvShape cs;
    CHX_PROPAGATE(conv_shape(*x, *w, *params, *y, "ConvInteger", &cs));
    ConvDirectArgs a;
    fill_conv_args(*x, *w, *params, *y, cs, &a);
    a.x_zp = x_zero_point;
    if (w_zero_point) {
        CHX_PROPAGATE(check_tensor(w_zero_point, "ConvInteger w_zero_point"));
        CHX_REQUIRE(w_zero_point->dtype == w->dtype, "ConvInteger: w_zero_point must have the dtype of w");
        int64_t len, stride;
        CHX_PROPAGATE(param_vector(*w_zero_point, cs.OC, "ConvInteger w_zero_point", &len, &stride));
        a.w_zp = static_cast<const char*>(w_zero_point->data);
        a.w_zp_len = (int32_t)len;
        a.w_zp_stride = stride;
    }
    hipStream_t s = as_stream(stream);
    // (a recorded run takes a kernel without scratch memory: the weights of this entry point arrive with the call)
    const bool capturing = stream_is_capturing(s);
    // The packed kernel multiplies faster but costs some 70 us of host time per call (read-back of the zero points,
    // allocations, packing): the two meet at 8 G multiply-adds, and it takes channels-last results only.
    const double macs = (double)a.total * cs.Cg * cs.KH * cs.KW;
    const bool packed = weights_fit_mfma(*w, params->group) && macs >= 0x1p33 && x_is_mfma_ready(*x);
    const bool product_first = cs.KH * cs.KW == 1 && (capturing || !packed || !faster_packed(*params, cs, a));
    auto product = [&](bool any) { return run_conv_as_product(*x, *w, x_zero_point, *params, cs, a, *y, any, s); };
    if (product_first) {
        const int rc = product(capturing);
        if (rc != CHX_HIP_EUNSUPPORTED) return rc;
    }
    if (!capturing && !packed) {
        int rc = run_conv_strip(a, s);
        if (rc == CHX_HIP_EUNSUPPORTED) rc = run_conv_planar(a, s);
        if (rc == CHX_HIP_EUNSUPPORTED) rc = product(true);
        if (rc != CHX_HIP_EUNSUPPORTED) return rc;
    }
    if (weights_fit_mfma(*w, params->group) && !capturing) {
        bool zero = true;
        if (w_zero_point) {
            std::vector<uint8_t> zp;
            CHX_PROPAGATE(read_back(*w_zero_point, &zp, s));
            zero = all_zero(zp);
        }
        if (zero) {
            ConvCall c;
            memset(&c, 0, sizeof(c));
            c.opt = read_launch_options();
            c.x = x;
            c.y = y;
            c.p = params;
            c.cs = cs;
            c.x_zp = x_zero_point;
            c.out_int32 = true;
            PackedWeights pw;
            CHX_PROPAGATE(make_packed(*w, false, s, &pw));
            const int rc = run_conv_mfma(c, pw, s);
            release_packed(&pw, false, s);
            if (rc != CHX_HIP_EUNSUPPORTED) return rc;
        }
    }
    const int rc = product(true);  // (zero points of the filters that are not 0)
    if (rc != CHX_HIP_EUNSUPPORTED) return rc;
    return launch_conv_direct(a, false, s);
}

extern "C" int chx_hip_matmul_integer(
        const chx_hip_tensor* a, const chx_hip_tensor* b, const chx_hip_tensor* a_zero_point,
        const chx_hip_tensor* b_zero_point, chx_hip_tensor* y, void* stream) {
    CHX_PROPAGATE(check_tensor(a, "MatMulInteger a"));
    CHX_PROPAGATE(check_tensor(b, "MatMulInteger b"));
    CHX_PROPAGATE(check_tensor(y, "MatMulInteger y"));
    CHX_REQUIRE(is_q8(a->dtype) && is_q8(b->dtype), "MatMulInteger: a and b must be uint8 or int8");
    CHX_REQUIRE(y->dtype == CHX_HIP_INT32, "MatMulInteger: y must be int32, got %s", dtype_name(y->dtype));
    MatMulShape ms;
    CHX_PROPAGATE(matmul_shape(*a, *b, *y, "MatMulInteger", &ms));
    MatMulDirectArgs m;
    fill_matmul_args(*a, *b, *y, ms, &m);
    if (a_zero_point) {
        CHX_PROPAGATE(check_tensor(a_zero_point, "MatMulInteger a_zero_point"));
        CHX_REQUIRE(is_q8(a_zero_point->dtype), "MatMulInteger: a_zero_point must be uint8 or int8");
        int64_t len, stride;
        CHX_PROPAGATE(param_vector(*a_zero_point, ms.K, "MatMulInteger a_zero_point", &len, &stride));  // CHECK_GE(1, ndim)
        m.a_zp = static_cast<const char*>(a_zero_point->data);
        m.a_zp_len = (int32_t)len;
        m.a_zp_stride = stride;
        m.a_zp_signed = a_zero_point->dtype == CHX_HIP_INT8;
    }
    if (b_zero_point) {
        CHX_PROPAGATE(check_tensor(b_zero_point, "MatMulInteger b_zero_point"));
        CHX_REQUIRE(is_q8(b_zero_point->dtype), "MatMulInteger: b_zero_point must be uint8 or int8");
        int64_t len, stride;
        CHX_PROPAGATE(param_vector(*b_zero_point, ms.N, "MatMulInteger b_zero_point", &len, &stride));
        m.b_zp = static_cast<const char*>(b_zero_point->data);
        m.b_zp_len = (int32_t)len;
        m.b_zp_stride = stride;
        m.b_zp_signed = b_zero_point->dtype == CHX_HIP_INT8;
    }
    hipStream_t s = as_stream(stream);
    const int rc = launch_matmul_i8(m, false, s);
    if (rc != CHX_HIP_EUNSUPPORTED) return rc;
    return launch_matmul_direct(m, false, s);
}

extern "C" int chx_hip_qlinear_matmul(
        const chx_hip_tensor* a, float a_scale, int32_t a_zero_point, const chx_hip_tensor* b, float b_scale,
        int32_t b_zero_point, float y_scale, int32_t y_zero_point, const chx_hip_tensor* bias, uint32_t flags,
        chx_hip_tensor* y, void* stream) {
    CHX_PROPAGATE(check_tensor(a, "QLinearMatMul a"));
    CHX_PROPAGATE(check_tensor(b, "QLinearMatMul b"));
    CHX_PROPAGATE(check_tensor(y, "QLinearMatMul y"));
    CHX_REQUIRE(is_q8(a->dtype) && is_q8(b->dtype), "QLinearMatMul: a and b must be uint8 or int8");
    MatMulShape ms;
    CHX_PROPAGATE(matmul_shape(*a, *b, *y, "QLinearMatMul", &ms));
    MatMulDirectArgs m;
    fill_matmul_args(*a, *b, *y, ms, &m);
    m.a_zp_imm = a_zero_point;
    m.b_zp_imm = b_zero_point;
    m.requant = 1;
    m.b_scale = b_scale;
    // the extension's bias is always the ONNX kind: int32, added to the accumulator
    CHX_PROPAGATE(fill_requant(a_scale, y_scale, y_zero_point, *y, bias, ms.N, flags | CHX_HIP_BIAS_ONNX_INT32,
                               "QLinearMatMul", &m.rq, &m.bias));
    hipStream_t s = as_stream(stream);
    const bool rne = (flags & CHX_HIP_ROUND_ONNX_RNE) != 0;
    const int rc = launch_matmul_i8(m, rne, s);
    if (rc != CHX_HIP_EUNSUPPORTED) return rc;
    return launch_matmul_direct(m, rne, s);
}

// ---- blocks of convolutions as one launch ------------------------------------------------------

namespace chx {
namespace {
// The operands of a convolution of a block: int8 weights, one scale or one per filter, an int32 bias on all of the block's or on none.
int check_block_operands(const chx_hip_conv_operands& c, bool biased, const char* what) {
    auto refuse = [&](const char* why) {
        set_error("%s: %s", what, why);
        return (int)CHX_HIP_EUNSUPPORTED;
    };
    CHX_PROPAGATE(check_tensor(c.w, what));
    CHX_PROPAGATE(check_tensor(c.w_scale, what));
    CHX_PROPAGATE(check_tensor(c.w_zero_point, what));
    if (c.w->ndim != 4 || c.w->dtype != CHX_HIP_INT8 || c.w_scale->dtype != CHX_HIP_FLOAT32 || c.w_scale->ndim > 1 || c.w_zero_point->dtype != CHX_HIP_INT8) return refuse("the type of an operand");
    const int64_t scales = numel(*c.w_scale);
    if (scales != 1 && scales != c.w->shape[0]) return refuse("the number of scales");
    if (c.bias) {
        CHX_PROPAGATE(check_tensor(c.bias, what));
        if (c.bias->dtype != CHX_HIP_INT32 || c.bias->ndim != 1 || c.bias->shape[0] != c.w->shape[0]) return refuse("a bias");
    }
    if ((c.bias != nullptr) != biased) return refuse("a bias on some of the convolutions");
    return CHX_HIP_OK;
}
}  // namespace
}  // namespace chx

// ---- inverted residual blocks ------------------------------------------------------------------

struct chx_hip_inverted_residual {
    int32_t channels = 0, out_channels = 0, stride = 1;
    bool has_bias = false, affine_residual = true;
    int device = 0;  // whose memory the operands are laid out in
    int tiles = 0, tiles_padded = 0, steps = 0, tiles_oc = 0;
    char* memory = nullptr;
    size_t at_w3 = 0, at_t1 = 0, at_t2 = 0, at_t3 = 0;
    std::mutex mutex;  // of `searched`
    std::vector<chx::SearchedResidual> searched;
};

extern "C" void chx_hip_inverted_residual_destroy(chx_hip_inverted_residual* plan) {
    if (!plan) return;
    (void)hipFree(plan->memory);
    delete plan;
}

extern "C" int chx_hip_inverted_residual_create(const chx_hip_conv_operands* stages, int32_t stride, void* stream, chx_hip_inverted_residual** out) {
    CHX_REQUIRE(stages != nullptr && out != nullptr, "inverted residual: null argument");
    *out = nullptr;
    auto refuse = [](const char* why) {
        set_error("inverted residual: %s", why);
        return (int)CHX_HIP_EUNSUPPORTED;
    };
    hipStream_t s = as_stream(stream);
    for (int i = 0; i < 3; ++i) CHX_PROPAGATE(check_block_operands(stages[i], stages[0].bias != nullptr, "inverted residual"));
    const chx_hip_tensor &w1 = *stages[0].w, &w2 = *stages[1].w, &w3 = *stages[2].w;
    const int64_t hid = w1.shape[0];
    if (w1.shape[2] != 1 || w1.shape[3] != 1 || w3.shape[2] != 1 || w3.shape[3] != 1 || w2.shape[2] != 3 || w2.shape[3] != 3 || w2.shape[1] != 1 || w2.shape[0] != hid ||
        w3.shape[1] != hid || (stride != 1 && stride != 2))
        return refuse("not 1x1, depthwise 3x3, 1x1");
    if (w1.shape[1] < 1 || w1.shape[1] > kInvertedMaxIn || hid < 1 || hid > 4096 || w3.shape[0] < 1 || w3.shape[0] > kInvertedMaxOut) return refuse("the number of channels");
    for (int i = 0; i < 3; ++i) {
        std::vector<uint8_t> zp;
        CHX_PROPAGATE(read_back(*stages[i].w_zero_point, &zp, s));
        if (!all_zero(zp)) return refuse("zero points of the weights");
    }
    std::unique_ptr<chx_hip_inverted_residual, void (*)(chx_hip_inverted_residual*)> p(new chx_hip_inverted_residual(), chx_hip_inverted_residual_destroy);
    CHX_HIP_CALL(hipGetDevice(&p->device));
    p->channels = (int32_t)w1.shape[1];
    p->out_channels = (int32_t)w3.shape[0];
    p->stride = stride;
    p->has_bias = stages[0].bias != nullptr;
    p->affine_residual = read_launch_options().affine_residual;
    p->tiles = (int)((hid + 31) / 32);
    p->tiles_padded = (p->tiles + 7) / 8 * 8;  // (the kernel takes up to eight at a time)
    p->steps = p->channels <= 32 ? 1 : p->channels <= 96 ? 3 : 5;
    p->tiles_oc = (p->out_channels + 31) / 32;
    p->at_w3 = (size_t)p->tiles_padded * p->steps * 1024;
    p->at_t1 = p->at_w3 + (size_t)p->tiles_padded * p->tiles_oc * 1024;
    p->at_t2 = p->at_t1 + (size_t)p->tiles_padded * 32 * 16;
    p->at_t3 = p->at_t2 + (size_t)p->tiles_padded * 32 * 32;
    CHX_PROPAGATE(spare_memory(reinterpret_cast<void**>(&p->memory), p->at_t3 + (size_t)p->tiles_oc * 32 * 16, "inverted residual"));
    auto table = [&](size_t at) { return reinterpret_cast<int32_t*>(p->memory + at); };
    CHX_PROPAGATE(pack_inverted_point(w1, *stages[0].w_scale, stages[0].bias, false, p->tiles_padded, p->steps, p->memory, table(p->at_t1), s));
    CHX_PROPAGATE(pack_inverted_depthwise(w2, *stages[1].w_scale, stages[1].bias, p->tiles_padded, table(p->at_t2), s));
    CHX_PROPAGATE(pack_inverted_point(w3, *stages[2].w_scale, stages[2].bias, true, p->tiles_oc, p->tiles_padded, p->memory + p->at_w3, table(p->at_t3), s));
    // (later calls may come on any stream)
    CHX_HIP_CALL(hipStreamSynchronize(s));
    *out = p.release();
    return CHX_HIP_OK;
}

extern "C" int chx_hip_inverted_residual_run(
        chx_hip_inverted_residual* plan, const chx_hip_tensor* x, float x_scale, int32_t x_zero_point, const float* y_scales, const int32_t* y_zero_points,
        int32_t y_dtype, uint32_t flags, const chx_hip_tensor* r, float r_scale, int32_t r_zero_point, float out_scale, int32_t out_zero_point, int32_t relu,
        chx_hip_tensor* out, void* stream) {
    CHX_REQUIRE(plan != nullptr && y_scales != nullptr && y_zero_points != nullptr, "inverted residual: null argument");
    CHX_PROPAGATE(check_tensor(x, "inverted residual x"));
    chx_hip_tensor outv;
    bool out_minus_128 = false;
    CHX_PROPAGATE(result_view(out, flags, "inverted residual out", &outv, &out_minus_128));
    auto refuse = [](const char* why) {
        set_error("inverted residual: %s", why);
        return (int)CHX_HIP_EUNSUPPORTED;
    };
    int device = 0;
    CHX_HIP_CALL(hipGetDevice(&device));
    if (device != plan->device) return refuse("another device than the one that it was created on");
    auto in_range = [](int32_t zp, int32_t dt) { return dt == CHX_HIP_INT8 ? zp >= -128 && zp <= 127 : zp >= 0 && zp <= 255; };
    if (x->ndim != 4 || out->ndim != 4 || !is_q8(x->dtype) || x->shape[1] != plan->channels || !in_range(x_zero_point, x->dtype)) return refuse("x");
    if ((flags & (CHX_HIP_ROUND_ONNX_RNE | CHX_HIP_FUSE_RELU)) != 0 || (plan->has_bias && !(flags & CHX_HIP_BIAS_ONNX_INT32))) return refuse("the flags");
    const int32_t out_dtype = r ? outv.dtype : y_dtype;
    if (y_dtype != CHX_HIP_UINT8 || outv.dtype != CHX_HIP_UINT8) return refuse("the type of a result");
    const int64_t N = x->shape[0], H = x->shape[2], W = x->shape[3], OH = (H - 1) / plan->stride + 1, OW = (W - 1) / plan->stride + 1;
    if (N < 1 || H < 1 || W < 1 || out->shape[0] != N || out->shape[1] != plan->out_channels || out->shape[2] != OH || out->shape[3] != OW) return refuse("the shape of the result");
    int64_t x_px = 0, o_px = 0, r_px = 0;
    if (!y_is_pixel_major(*x, &x_px) || !y_is_pixel_major(outv, &o_px)) return refuse("x or out is not channels-last");
    const int64_t chunks = (plan->channels + 15) / 16;
    if (!aligned(x->data, 16) || x_px % 16 != 0 || x_px < 16 * chunks || !aligned(out->data, 16) || o_px % 16 != 0 || o_px < plan->out_channels) return refuse("pixels that are not whole 16-byte chunks");
    if (H * W * x_px >= (int64_t(1) << 31) || N >= (int64_t(1) << 24)) return refuse("an image of 2 GB");
    if (byte_ranges_overlap(outv, *x)) return refuse("out overlaps x");
    InvertedResidualArgs a;
    memset(&a, 0, sizeof(a));
    for (int i = 0; i < 3; ++i) {
        if (!in_range(y_zero_points[i], CHX_HIP_UINT8)) return refuse("a zero point");
    }
    auto product = [&](int i, bool two_fma) {
        const QuantParams q = make_quant_params(y_scales[i], y_zero_points[i], false);
        return product_form(q, q.lo, false, two_fma);
    };
    a.q1 = product(0, true);
    a.q2 = product(1, true);
    if (a.q1.path != a.q2.path) {
        a.q1 = product(0, false);
        a.q2 = product(1, false);
    }
    a.q3 = product(2, true);
    if (a.q1.path != a.q2.path || (a.q1.path != 1 && a.q1.path != 3) || a.q3.path == 0) return refuse("a requantization without a product form");
    hipStream_t s = as_stream(stream);
    if (r) {
        CHX_PROPAGATE(check_tensor(r, "inverted residual r"));
        for (int i = 0; i < 4; ++i)
            if (r->ndim != 4 || r->shape[i] != out->shape[i]) return refuse("the shape of r");
        if (!is_q8(r->dtype) || !in_range(r_zero_point, r->dtype) || !in_range(out_zero_point, out_dtype) || !(out_scale >= 0x1p-60f && out_scale <= 0x1p60f)) return refuse("the quantization of the sum");
        if (!y_is_pixel_major(*r, &r_px) || !aligned(r->data, 16) || r_px % 16 != 0 || r_px < plan->out_channels) return refuse("r is not channels-last in whole chunks");
        if (byte_ranges_overlap(outv, *r)) return refuse("out overlaps r");
    }
    a.N = (int32_t)N; a.H = (int32_t)H; a.W = (int32_t)W; a.OH = (int32_t)OH; a.OW = (int32_t)OW;
    a.OC = plan->out_channels;
    a.hid_tiles = plan->tiles;
    a.hid_tiles_padded = plan->tiles_padded;
    a.x_chunks = (int32_t)chunks;
    a.KS = plan->steps;
    CHX_PROPAGATE(plan_inverted_residual(&a, plan->stride));
    if (r) {  // (the first call with a sum's parameters launches a search: nothing is refused behind it)
        std::lock_guard<std::mutex> lock(plan->mutex);
        CHX_PROPAGATE(residual_of(*r, r_px, y_scales[2], y_zero_points[2], y_dtype, r_scale, r_zero_point, out_scale, out_zero_point, out_dtype, relu != 0,
                                  plan->affine_residual, &plan->searched, s, &a.res));
    }
    a.x = static_cast<const char*>(x->data);
    a.y = static_cast<char*>(out->data);
    a.x_px = x_px;
    a.x_n = H * W * x_px;
    a.y_px = o_px;
    a.y_n = OH * OW * o_px;
    a.w1 = plan->memory;
    a.w3 = plan->memory + plan->at_w3;
    a.t1 = reinterpret_cast<const int32_t*>(plan->memory + plan->at_t1);
    a.t2 = reinterpret_cast<const int32_t*>(plan->memory + plan->at_t2);
    a.t3 = reinterpret_cast<const int32_t*>(plan->memory + plan->at_t3);
    a.x_flip = x->dtype == CHX_HIP_UINT8 ? 0x80808080u : 0u;
    a.y_flip = out_minus_128 ? 0x80808080u : 0u;
    a.corr1 = (x->dtype == CHX_HIP_UINT8 ? 128 : 0) - x_zero_point;
    a.corr2 = 128 - y_zero_points[0];
    a.corr3 = 128 - y_zero_points[1];
    a.s1 = x_scale;
    a.s2 = y_scales[0];
    a.s3 = y_scales[1];
    a.fill = (int32_t)(((uint32_t)y_zero_points[0] ^ 0x80u) * 0x01010101u);
    return launch_inverted_residual(a, plan->stride, s);
}

// ---- bottleneck blocks -------------------------------------------------------------------------

struct chx_hip_bottleneck {
    int32_t mid = 0, wide = 0, next = 0;
    bool has_bias = false, affine_residual = true;
    int device = 0;  // whose memory the operands are laid out in
    char* memory = nullptr;
    size_t at[3] = {0, 0, 0}, at_table = 0;
    std::mutex mutex;  // of `searched`
    std::vector<chx::SearchedResidual> searched;
};

extern "C" void chx_hip_bottleneck_destroy(chx_hip_bottleneck* plan) {
    if (!plan) return;
    (void)hipFree(plan->memory);
    delete plan;
}

extern "C" int chx_hip_bottleneck_create(const chx_hip_conv_operands* stages, int32_t count, void* stream, chx_hip_bottleneck** out) {
    CHX_REQUIRE(stages != nullptr && out != nullptr && (count == 2 || count == 3), "bottleneck: null argument");
    *out = nullptr;
    auto refuse = [](const char* why) {
        set_error("bottleneck: %s", why);
        return (int)CHX_HIP_EUNSUPPORTED;
    };
    hipStream_t s = as_stream(stream);
    int64_t channels = 0;
    for (int i = 0; i < count; ++i) {
        CHX_PROPAGATE(check_block_operands(stages[i], stages[0].bias != nullptr, "bottleneck"));
        const chx_hip_tensor& w = *stages[i].w;
        const int64_t k = i == 0 ? 3 : 1;
        if (w.shape[2] != k || w.shape[3] != k || (i > 0 && w.shape[1] != channels)) return refuse("not 3x3, 1x1, 1x1");
        channels = w.shape[0];
    }
    const int64_t mid = stages[0].w->shape[0], wide = stages[1].w->shape[0], next = count == 3 ? channels : 0;
    if (stages[0].w->shape[1] != mid || !bottleneck_takes_channels(mid, wide, next)) return refuse("the number of channels");
    for (int i = 0; i < count; ++i) {
        std::vector<uint8_t> zp;
        CHX_PROPAGATE(read_back(*stages[i].w_zero_point, &zp, s));
        if (!all_zero(zp)) return refuse("zero points of the weights");
    }
    std::unique_ptr<chx_hip_bottleneck, void (*)(chx_hip_bottleneck*)> p(new chx_hip_bottleneck(), chx_hip_bottleneck_destroy);
    CHX_HIP_CALL(hipGetDevice(&p->device));
    p->mid = (int32_t)mid;
    p->wide = (int32_t)wide;
    p->next = (int32_t)next;
    p->has_bias = stages[0].bias != nullptr;
    p->affine_residual = read_launch_options().affine_residual;
    p->at[1] = (size_t)(9 * mid * mid);
    p->at[2] = p->at[1] + (size_t)(mid * wide);
    p->at_table = p->at[2] + (size_t)(wide * next);
    CHX_PROPAGATE(spare_memory(reinterpret_cast<void**>(&p->memory), p->at_table + (size_t)round_up(mid + wide + next, 64) * 16, "bottleneck"));  // (the kernel reads 64 rows at a time)
    int32_t* table = reinterpret_cast<int32_t*>(p->memory + p->at_table);
    for (int i = 0; i < count; ++i) {
        CHX_PROPAGATE(pack_bottleneck(*stages[i].w, *stages[i].w_scale, stages[i].bias, p->memory + p->at[i], table, s));
        table += 4 * stages[i].w->shape[0];
    }
    // (later calls may come on any stream)
    CHX_HIP_CALL(hipStreamSynchronize(s));
    *out = p.release();
    return CHX_HIP_OK;
}

namespace chx {
namespace {
// The launch of a block over so many pixels.
int plan_bottleneck_of(const chx_hip_bottleneck& plan, int64_t N, int64_t H, int64_t W, BottleneckArgs* a) {
    if (N < 1 || H < 1 || W < 1 || N > INT32_MAX || H > INT32_MAX || W > INT32_MAX || N * H >= (int64_t(1) << 30) || N * H * W >= (int64_t(1) << 30))
        CHX_FAIL(CHX_HIP_EUNSUPPORTED, "bottleneck: the number of pixels");
    memset(a, 0, sizeof(*a));
    a->pixels = (int32_t)(N * H * W);
    a->H = (int32_t)H;
    a->W = (int32_t)W;
    a->mid = plan.mid;
    a->wide = plan.wide;
    a->next = plan.next;
    return plan_bottleneck(a);
}
}  // namespace
}  // namespace chx

extern "C" int chx_hip_bottleneck_takes(const chx_hip_bottleneck* plan, int64_t n, int64_t h, int64_t w) {
    CHX_REQUIRE(plan != nullptr, "bottleneck: null plan");
    BottleneckArgs a;
    return plan_bottleneck_of(*plan, n, h, w, &a);
}

extern "C" int chx_hip_bottleneck_run(
        chx_hip_bottleneck* plan, const chx_hip_tensor* x, float x_scale, int32_t x_zero_point, const float* y_scales, const int32_t* y_zero_points, int32_t y_dtype,
        uint32_t flags, const chx_hip_tensor* r, float r_scale, int32_t r_zero_point, float out_scale, int32_t out_zero_point, int32_t relu, uint32_t out_flags, chx_hip_tensor* out,
        uint32_t next_flags, chx_hip_tensor* next, void* stream) {
    CHX_REQUIRE(plan != nullptr && y_scales != nullptr && y_zero_points != nullptr && (next != nullptr) == (plan->next != 0), "bottleneck: null argument");
    CHX_PROPAGATE(check_tensor(x, "bottleneck x"));
    CHX_PROPAGATE(check_tensor(r, "bottleneck r"));
    chx_hip_tensor views[2];
    chx_hip_tensor* const results[2] = {out, next};
    bool minus_128[2] = {false, false};
    CHX_PROPAGATE(result_view(out, out_flags, "bottleneck out", &views[0], &minus_128[0]));
    if (next) CHX_PROPAGATE(result_view(next, next_flags, "bottleneck next", &views[1], &minus_128[1]));
    auto refuse = [](const char* why) {
        set_error("bottleneck: %s", why);
        return (int)CHX_HIP_EUNSUPPORTED;
    };
    int device = 0;
    CHX_HIP_CALL(hipGetDevice(&device));
    if (device != plan->device) return refuse("another device than the one that it was created on");
    auto in_range = [](int32_t zp, int32_t dt) { return dt == CHX_HIP_INT8 ? zp >= -128 && zp <= 127 : zp >= 0 && zp <= 255; };
    if (x->ndim != 4 || !is_q8(x->dtype) || x->shape[1] != plan->mid || !in_range(x_zero_point, x->dtype)) return refuse("x");
    if ((flags & (CHX_HIP_ROUND_ONNX_RNE | CHX_HIP_FUSE_RELU)) != 0 || (plan->has_bias && !(flags & CHX_HIP_BIAS_ONNX_INT32))) return refuse("the flags");
    if (y_dtype != CHX_HIP_UINT8) return refuse("the type of a result");
    const int64_t N = x->shape[0], H = x->shape[2], W = x->shape[3];
    BottleneckArgs a;
    CHX_PROPAGATE(plan_bottleneck_of(*plan, N, H, W, &a));
    const int64_t most_px = int64_t(1) << 24;  // (bytes from a pixel to the next: 24-bit products)
    int64_t x_px = 0, px[2] = {0, 0}, r_px = 0;
    if (!y_is_pixel_major(*x, &x_px) || !aligned(x->data, 16) || x_px % 16 != 0 || x_px >= most_px) return refuse("x is not channels-last in whole chunks");
    for (int i = 0; i < (next ? 2 : 1); ++i) {
        const chx_hip_tensor& t = *results[i];
        if (t.ndim != 4 || t.shape[0] != N || t.shape[1] != (i ? plan->next : plan->wide) || t.shape[2] != H || t.shape[3] != W) return refuse("the shape of a result");
        if (views[i].dtype != CHX_HIP_UINT8) return refuse("the type of a result");
        if (!y_is_pixel_major(views[i], &px[i]) || !aligned(t.data, 16) || px[i] % 16 != 0 || px[i] >= most_px) return refuse("a result is not channels-last in whole chunks");
        if (byte_ranges_overlap(views[i], *x) || byte_ranges_overlap(views[i], *r)) return refuse("a result overlaps an operand");
    }
    if (next && byte_ranges_overlap(views[0], views[1])) return refuse("the results overlap");
    for (int i = 0; i < 4; ++i)
        if (r->ndim != 4 || r->shape[i] != out->shape[i]) return refuse("the shape of r");
    if (!is_q8(r->dtype) || !in_range(r_zero_point, r->dtype) || !in_range(out_zero_point, CHX_HIP_UINT8) || !(out_scale >= 0x1p-60f && out_scale <= 0x1p60f)) return refuse("the quantization of the sum");
    if (!y_is_pixel_major(*r, &r_px) || !aligned(r->data, 16) || r_px % 16 != 0 || r_px >= most_px) return refuse("r is not channels-last in whole chunks");
    QuantProduct* const products[3] = {&a.q1, &a.q2, &a.q3};
    for (int i = 0; i < (next ? 3 : 2); ++i) {
        if (!in_range(y_zero_points[i], CHX_HIP_UINT8)) return refuse("a zero point");
        const QuantParams q = make_quant_params(y_scales[i], y_zero_points[i], false);
        *products[i] = product_form(q, q.lo, false, true);
        if (products[i]->path != 1 && products[i]->path != 3) return refuse("a requantization without a product form");
    }
    hipStream_t s = as_stream(stream);
    {  // (the first call with a sum's parameters launches a search: nothing is refused behind it)
        std::lock_guard<std::mutex> lock(plan->mutex);
        CHX_PROPAGATE(residual_of(*r, r_px, y_scales[1], y_zero_points[1], y_dtype, r_scale, r_zero_point, out_scale, out_zero_point, CHX_HIP_UINT8, relu != 0, plan->affine_residual,
                                  &plan->searched, s, &a.res));
    }
    a.x = static_cast<const char*>(x->data);
    a.y = static_cast<char*>(out->data);
    a.z = next ? static_cast<char*>(next->data) : nullptr;
    a.x_px = x_px;
    a.y_px = px[0];
    a.z_px = px[1];
    a.w1 = plan->memory;
    a.w2 = plan->memory + plan->at[1];
    a.w3 = plan->memory + plan->at[2];
    a.table = reinterpret_cast<const int32_t*>(plan->memory + plan->at_table);
    a.x_flip = x->dtype == CHX_HIP_UINT8 ? 0x80808080u : 0u;
    a.y_flip = minus_128[0] ? 0x80808080u : 0u;
    a.z_flip = minus_128[1] ? 0x80808080u : 0u;
    a.corr1 = (x->dtype == CHX_HIP_UINT8 ? 128 : 0) - x_zero_point;
    a.corr2 = 128 - y_zero_points[0];
    a.corr3 = 128 - out_zero_point;
    a.s1 = x_scale;
    a.s2 = y_scales[0];
    a.s3 = out_scale;
    a.fill = (int32_t)(((uint32_t)x_zero_point ^ (x->dtype == CHX_HIP_UINT8 ? 0x80u : 0u)) & 0xffu) * 0x01010101;
    return launch_bottleneck(a, s);
}
