// Library state, error reporting and the thin device-memory helpers of the C ABI.
#include <cmath>
#include <cstring>
#include <mutex>
#include <unordered_map>

#include "chx_internal.h"
#include "quant_math.h"

namespace chx {

// Where the codes of one quantization begin: below[k] is the last float whose code is less than k, the float after it
// (above(below[k], 1)) the first whose code is k or more.
struct CodeBounds {
    float below[256], from[256];
};

// n floats above v (which is that far from 0)
static float above(float v, int n) {
    int32_t bits;
    memcpy(&bits, &v, 4);
    bits += bits < 0 ? -n : n;
    memcpy(&v, &bits, 4);
    return v;
}

// The reference's QuantizeLinear in front of the conversion, which takes the floor and saturates.
static float reference_form(float v, const QuantParams& q) {
    const float s = v / q.scale, u = s + q.zpf;
    return u + 0.5f;
}

static bool find_bounds(const QuantParams& q, CodeBounds* b) {
    if (!(q.scale > 1e-30f && q.scale < 1e30f)) return false;
    for (int k = 1; k <= 255; ++k) {
        const float at = (float)k, v = (float)(((double)k - 0.5 - (double)q.zpf) * (double)q.scale);
        int lo = -1024, hi = 1024;  // the additions round by at most 2^-16, which is 512 floats at 0.5
        if (!(reference_form(above(v, lo), q) < at && reference_form(above(v, hi), q) >= at)) return false;
        while (hi - lo > 1) {
            const int mid = (lo + hi) / 2;
            (reference_form(above(v, mid), q) < at ? lo : hi) = mid;
        }
        b->below[k] = above(v, lo);
        b->from[k] = above(v, hi);
    }
    return true;
}

static float product_of(float v, const QuantProduct& p) {
    return p.path == 3 ? std::fma(v, p.inv, std::fma(v, p.inv_low, p.half)) : std::fma(v, p.inv, v * p.inv_low) + p.half;
}

static bool same_codes(const CodeBounds& b, const QuantProduct& p) {
    for (int k = 1; k <= 255; ++k)
        if (!(product_of(b.below[k], p) < (float)k && product_of(b.from[k], p) >= (float)k)) return false;
    // The inner sum of path 3 moves in steps of 2^-25 and against v where inv_low is negative.  From a quotient of 0.5 up
    // the product grows by as much from one float to the next; from 0.25 up it does over two; below that no t reaches 1.
    for (int n = 1; n <= 8; ++n)
        if (!(product_of(above(b.below[1], -n), p) < 1.f && product_of(above(b.from[1], n), p) >= 1.f)) return false;
    return true;
}

// inv moved by `ulps` and half by `half_ulps`
static QuantProduct product_with(const QuantParams& q, int path, int ulps, int half_ulps) {
    QuantProduct p = {};
    p.path = path;
    p.inv = above(1.0f / q.scale, ulps);
    p.inv_low = (float)(1.0 / (double)q.scale - (double)p.inv);
    p.half = above(q.zpf + 0.5f, half_ulps);
    return p;
}

// Path 1 for values that may be infinite: inv below the reciprocal and inv_low above 0, so that the two products of an
// infinity have one sign.
static QuantProduct product_below(const QuantParams& q) {
    QuantProduct p = product_with(q, 1, 0, 0);
    if (p.inv_low < 0.f) p = product_with(q, 1, -1, 0);
    if (p.inv_low == 0.f) p.inv_low = p.inv * 0x1p-60f;
    return p;
}

// The short forms of one quantization (path 0: there is none).
struct ProductForms {
    QuantProduct plain, two_fma, any_value;
};

static ProductForms find_forms(const QuantParams& q) {
    ProductForms f = {};
    CodeBounds b;
    if (!find_bounds(q, &b)) return f;
    const QuantProduct p = product_with(q, 1, 0, 0);
    if (same_codes(b, p)) f.plain = p;
    const QuantProduct below = product_below(q);
    if (below.inv_low > 0.f && same_codes(b, below)) f.any_value = below;
    // (99 of 100 scales have one in this range, most within a few steps)
    for (int i = 0; q.zpf == 0.f && i < 129 * 7 && f.two_fma.path == 0; ++i) {
        const int ring = (i / 7 + 1) / 2;
        const QuantProduct t = product_with(q, 3, (i / 7) & 1 ? ring : -ring, i % 7 - 3);
        if (same_codes(b, t)) f.two_fma = t;
    }
    return f;
}

// Finding them takes about 25 us, for each of a network's layers: the process remembers them by scale and zero point, for
// every plan, plan-less call and thread.  (A ResNet-50 has 54 pairs; a table of 256 places found by a hash alone had
// four of them evict each other: a pass through the 54 took 283 us of host time instead of 136.)  2000 pairs are some 200 KB; more start over.
static ProductForms known_forms(const QuantParams& q) {
    static std::mutex* mutex = new std::mutex;  // (never destroyed: calls may come from other destructors)
    static auto* known = new std::unordered_map<uint64_t, ProductForms>;
    uint32_t scale, zp;
    memcpy(&scale, &q.scale, 4);
    memcpy(&zp, &q.zpf, 4);
    const uint64_t key = (uint64_t)scale << 32 | zp;
    {
        std::lock_guard<std::mutex> lock(*mutex);
        const auto it = known->find(key);
        if (it != known->end()) return it->second;
    }
    const ProductForms f = find_forms(q);
    std::lock_guard<std::mutex> lock(*mutex);
    if (known->size() >= 2000) known->clear();
    (*known)[key] = f;
    return f;
}

QuantProduct product_form(const QuantParams& q, float lo_folded, bool rne, bool two_fma) {
    if (rne || q.lo != 0.f || q.hi != 255.f) return QuantProduct{};
    const ProductForms f = known_forms(q);
    const bool bound = lo_folded > 0.f;
    QuantProduct p = two_fma && !bound && f.two_fma.path != 0 ? f.two_fma : f.plain;
    if (p.path == 1 && bound) p.path = 2;
    p.floor_half = lo_folded + 0.5f;
    return p;
}

QuantProduct product_form_of_any_value(const QuantParams& q) {
    return q.lo != 0.f || q.hi != 255.f ? QuantProduct{} : known_forms(q).any_value;
}

static thread_local std::string g_last_error;

void set_error(const char* fmt, ...) {
    char buf[2048];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    g_last_error = buf;
}

bool host_libm_uses_fma() {
    static const bool v = [] {
        volatile float x = 0.0f;
        const uint32_t bits = 0x4202422fu;
        float xf;
        memcpy(&xf, &bits, 4);
        x = xf;
        const float e = expf(x);
        uint32_t eb;
        memcpy(&eb, &e, 4);
        return eb == 0x56fc9f1cu;  // 0x1.f93e38p+46: the fused-reduction result
    }();
    return v;
}

int check_tensor(const chx_hip_tensor* t, const char* what) {
    CHX_REQUIRE(t != nullptr, "%s: null tensor descriptor", what);
    CHX_REQUIRE(t->ndim >= 0 && t->ndim <= CHX_HIP_MAX_NDIM, "%s: ndim %d out of range", what, t->ndim);
    CHX_REQUIRE(dtype_size(t->dtype) != 0, "%s: unknown dtype code %d", what, t->dtype);
    int64_t n = 1;
    for (int i = 0; i < t->ndim; ++i) {
        CHX_REQUIRE(t->shape[i] >= 0, "%s: negative extent on axis %d", what, i);
        n *= t->shape[i];
    }
    CHX_REQUIRE(n == 0 || t->data != nullptr, "%s: null data pointer for %lld elements", what, (long long)n);
    return CHX_HIP_OK;
}

bool same_dense_layout(const chx_hip_tensor& a, const chx_hip_tensor& b) {
    if (!same_shape(a, b)) return false;
    if (is_contiguous(a) && is_contiguous(b)) return true;
    const int64_t ea = dtype_size(a.dtype), eb = dtype_size(b.dtype);
    // identical stride pattern in elements, and dense: sort axes by stride and check packing
    int order[CHX_HIP_MAX_NDIM];
    int nd = 0;
    for (int i = 0; i < a.ndim; ++i) {
        if (a.shape[i] == 1) continue;
        if (a.strides[i] % ea || b.strides[i] % eb) return false;
        if (a.strides[i] / ea != b.strides[i] / eb) return false;
        order[nd++] = i;
    }
    for (int i = 0; i < nd; ++i)
        for (int j = i + 1; j < nd; ++j)
            if (a.strides[order[j]] < a.strides[order[i]]) {
                int t = order[i];
                order[i] = order[j];
                order[j] = t;
            }
    int64_t expect = ea;
    for (int i = 0; i < nd; ++i) {
        if (a.strides[order[i]] != expect) return false;
        expect *= a.shape[order[i]];
    }
    return true;
}

int launch_check(const char* kernel) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) CHX_FAIL(CHX_HIP_ERUNTIME, "launch of %s failed: %s", kernel, hipGetErrorString(e));
    return CHX_HIP_OK;
}

int spare_memory(void** p, size_t bytes, const char* what) {
    const hipError_t e = hipMalloc(p, bytes);
    if (e == hipSuccess) return CHX_HIP_OK;
    *p = nullptr;
    (void)hipGetLastError();
    CHX_FAIL(e == hipErrorOutOfMemory ? CHX_HIP_EUNSUPPORTED : CHX_HIP_ERUNTIME, "%s: hipMalloc of %zu bytes failed: %s", what, bytes, hipGetErrorString(e));
}

bool stream_is_capturing(hipStream_t s) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &st) != hipSuccess) {
        (void)hipGetLastError();
        return true;  // when in doubt, behave as if it were
    }
    return st != hipStreamCaptureStatusNone;
}

int scratch_alloc(void** p, size_t bytes, hipStream_t s) {
    *p = nullptr;
    if (bytes == 0) return CHX_HIP_OK;
    // A stream-ordered allocation on a capturing stream would become a memory node of the graph, whose replays then
    // run kernels on addresses that are not mapped (a device fault).  Callers that may be captured keep their scratch
    // between calls (plans) or take a path without scratch.
    if (stream_is_capturing(s)) CHX_FAIL(CHX_HIP_EUNSUPPORTED, "scratch memory cannot be allocated while the stream is being captured into a graph");
    CHX_HIP_CALL(hipMallocAsync(p, bytes, s));
    return CHX_HIP_OK;
}

void scratch_free(void* p, hipStream_t s) {
    if (p) (void)hipFreeAsync(p, s);
}

namespace {
constexpr int kMostDevices = 16;
constexpr size_t kMostShared = size_t(256) << 20;
struct SharedBlock {
    std::mutex mutex;
    void* ptr = nullptr;
    size_t size = 0;
    int small_uses = 0;  // calls in a row that needed less than a quarter of the block
};
SharedBlock& shared_block(int device) {
    static SharedBlock* blocks = new SharedBlock[kMostDevices];  // never destroyed: calls may come from other destructors
    return blocks[device];
}
}  // namespace

int Scratch::acquire(size_t bytes, hipStream_t s) {
    int device = 0;
    if (s != nullptr || bytes > kMostShared || hipGetDevice(&device) != hipSuccess || device >= kMostDevices) {
        stream_ = s;
        return scratch_alloc(&ptr_, bytes, s);
    }
    SharedBlock& b = shared_block(device);
    b.mutex.lock();
    shared_ = device;
    b.small_uses = bytes * 4 < b.size ? b.small_uses + 1 : 0;
    if (bytes > b.size || b.small_uses > 256) {
        size_t size = size_t(1) << 20;
        while (size < bytes) size *= 2;
        if (b.ptr) CHX_HIP_CALL(hipFree(b.ptr));  // (waits for the work that still uses it)
        b.ptr = nullptr;
        b.size = 0;
        b.small_uses = 0;
        CHX_HIP_CALL(hipMalloc(&b.ptr, size));
        b.size = size;
    }
    ptr_ = b.ptr;
    return CHX_HIP_OK;
}

Scratch::~Scratch() {
    if (shared_ >= 0) shared_block(shared_).mutex.unlock();
    else scratch_free(ptr_, stream_);
}

}  // namespace chx

using namespace chx;

struct chx_hip_graph {
    hipGraphExec_t exec;
};

extern "C" {

const char* chx_hip_last_error(void) {
    return g_last_error.c_str();
}

const char* chx_hip_version(void) {
    return "chx_hip 0.1 (gfx950)";
}

int chx_hip_init(int device) {
    int count = 0;
    CHX_HIP_CALL(hipGetDeviceCount(&count));
    CHX_REQUIRE(device >= 0 && device < count, "device %d out of range (%d visible)", device, count);
    CHX_HIP_CALL(hipSetDevice(device));
    hipDeviceProp_t prop;
    CHX_HIP_CALL(hipGetDeviceProperties(&prop, device));
    if (strncmp(prop.gcnArchName, "gfx950", 6) != 0)
        CHX_FAIL(CHX_HIP_EUNSUPPORTED, "device %d is %s; this library holds gfx950 code only", device, prop.gcnArchName);
    return prepare_noalloc_scratch();
}

int chx_hip_get_device(int32_t* device) {
    CHX_REQUIRE(device != nullptr, "null output");
    int d = 0;
    CHX_HIP_CALL(hipGetDevice(&d));
    *device = d;
    return CHX_HIP_OK;
}

int chx_hip_get_device_props(chx_hip_device_props* out) {
    CHX_REQUIRE(out != nullptr, "null output");
    int dev = 0;
    CHX_HIP_CALL(hipGetDevice(&dev));
    hipDeviceProp_t prop;
    CHX_HIP_CALL(hipGetDeviceProperties(&prop, dev));
    memset(out, 0, sizeof(*out));
    out->compute_units = prop.multiProcessorCount;
    out->clock_khz = prop.clockRate;
    out->memory_clock_khz = prop.memoryClockRate;
    out->memory_bus_bits = prop.memoryBusWidth;
    out->total_memory = (int64_t)prop.totalGlobalMem;
    strncpy(out->arch, prop.gcnArchName, sizeof(out->arch) - 1);
    strncpy(out->name, prop.name, sizeof(out->name) - 1);
    return CHX_HIP_OK;
}

int chx_hip_malloc(void** ptr, size_t bytes) {
    CHX_REQUIRE(ptr != nullptr, "null output pointer");
    *ptr = nullptr;
    if (bytes == 0) return CHX_HIP_OK;
    CHX_HIP_CALL(hipMalloc(ptr, bytes));
    return CHX_HIP_OK;
}

int chx_hip_free(void* ptr) {
    if (ptr) CHX_HIP_CALL(hipFree(ptr));
    return CHX_HIP_OK;
}

int chx_hip_memcpy_h2d(void* dst, const void* src, size_t bytes, void* stream) {
    if (bytes == 0) return CHX_HIP_OK;
    CHX_REQUIRE(dst && src, "null pointer");
    CHX_HIP_CALL(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, as_stream(stream)));
    CHX_HIP_CALL(hipStreamSynchronize(as_stream(stream)));
    return CHX_HIP_OK;
}

int chx_hip_memcpy_d2h(void* dst, const void* src, size_t bytes, void* stream) {
    if (bytes == 0) return CHX_HIP_OK;
    CHX_REQUIRE(dst && src, "null pointer");
    int rc = CHX_HIP_OK;
    if (small_copy_to_host(dst, src, bytes, as_stream(stream), &rc)) return rc;
    CHX_HIP_CALL(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, as_stream(stream)));
    CHX_HIP_CALL(hipStreamSynchronize(as_stream(stream)));
    return CHX_HIP_OK;
}

int chx_hip_memset(void* dst, int value, size_t bytes, void* stream) {
    if (bytes == 0) return CHX_HIP_OK;
    CHX_REQUIRE(dst != nullptr, "null pointer");
    CHX_HIP_CALL(hipMemsetAsync(dst, value, bytes, as_stream(stream)));
    return CHX_HIP_OK;
}

int chx_hip_stream_synchronize(void* stream) {
    CHX_HIP_CALL(hipStreamSynchronize(as_stream(stream)));
    return CHX_HIP_OK;
}

int chx_hip_device_synchronize(void) {
    CHX_HIP_CALL(hipDeviceSynchronize());
    return CHX_HIP_OK;
}

int chx_hip_stream_create(void** stream) {
    CHX_REQUIRE(stream != nullptr, "null output");
    hipStream_t s = nullptr;
    CHX_HIP_CALL(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    *stream = s;
    return CHX_HIP_OK;
}

int chx_hip_stream_destroy(void* stream) {
    if (stream) CHX_HIP_CALL(hipStreamDestroy(as_stream(stream)));
    return CHX_HIP_OK;
}

int chx_hip_capture_begin(void* stream) {
    CHX_REQUIRE(stream != nullptr, "the null stream cannot be captured");
    // thread-local mode: calls of other threads (another program running eagerly) are not affected
    CHX_HIP_CALL(hipStreamBeginCapture(as_stream(stream), hipStreamCaptureModeThreadLocal));
    return CHX_HIP_OK;
}

int chx_hip_capture_end(void* stream, chx_hip_graph** graph) {
    CHX_REQUIRE(stream != nullptr && graph != nullptr, "null argument");
    *graph = nullptr;
    hipGraph_t g = nullptr;
    hipError_t e = hipStreamEndCapture(as_stream(stream), &g);
    if (e != hipSuccess || g == nullptr) {
        (void)hipGetLastError();
        if (g) (void)hipGraphDestroy(g);
        CHX_FAIL(CHX_HIP_ERUNTIME, "the capture did not give a graph: %s", hipGetErrorString(e));
    }
    hipGraphExec_t exec = nullptr;
    e = hipGraphInstantiate(&exec, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (e != hipSuccess) CHX_FAIL(CHX_HIP_ERUNTIME, "hipGraphInstantiate failed: %s", hipGetErrorString(e));
    chx_hip_graph* out = new chx_hip_graph();
    out->exec = exec;
    *graph = out;
    return CHX_HIP_OK;
}

int chx_hip_stream_is_capturing(void* stream) {
    if (!stream) return 0;
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(as_stream(stream), &st) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    return st != hipStreamCaptureStatusNone ? 1 : 0;
}

int chx_hip_graph_launch(const chx_hip_graph* graph, void* stream) {
    CHX_REQUIRE(graph != nullptr, "null graph");
    CHX_HIP_CALL(hipGraphLaunch(graph->exec, as_stream(stream)));
    return CHX_HIP_OK;
}

void chx_hip_graph_destroy(chx_hip_graph* graph) {
    if (!graph) return;
    (void)hipGraphExecDestroy(graph->exec);
    delete graph;
}

}  // extern "C"
