// Small results to the host.  A kernel writes them into pinned memory and then a sequence number the host polls: the
// host has 4 KB 8 us after the kernel before it ended, where a copy into pageable memory and a stream synchronization
// take 22 (64 KB: 13 against 45 us, 256 KB: 21 against 32; beyond 512 KB the copy engine wins).
#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstring>
#include <mutex>
#include <vector>

#include "chx_internal.h"

namespace chx {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v4i_u __attribute__((ext_vector_type(4), aligned(1)));

constexpr int kMaxRanges = 8;
constexpr size_t kMostBytes = 512 * 1024;
constexpr int kThreads = 256;

struct CopyOutArgs {
    const char* src[kMaxRanges];
    uint32_t bytes[kMaxRanges], at[kMaxRanges];  // `at`: where the range lies in the pinned block, a multiple of 16
    int32_t n;
    char* dst;
    uint32_t* arrived;  // device memory, 0 between launches
    uint32_t* flag;     // pinned
    uint32_t seq;
};

__global__ __launch_bounds__(kThreads) void copy_out_kernel(CopyOutArgs a) {
    for (int r = 0; r < a.n; ++r) {
        const uint32_t whole = a.bytes[r] / 16;
        char* dst = a.dst + a.at[r];
        for (uint32_t i = blockIdx.x * kThreads + threadIdx.x; i < whole; i += gridDim.x * kThreads)
            reinterpret_cast<v4i*>(dst)[i] = reinterpret_cast<const v4i_u*>(a.src[r])[i];
        if (blockIdx.x == 0 && threadIdx.x < a.bytes[r] % 16) dst[whole * 16 + threadIdx.x] = a.src[r][whole * 16 + threadIdx.x];
    }
    // every work-group's bytes are out before it counts itself in; the last one tells the host
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t before = __hip_atomic_fetch_add(a.arrived, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
        if (before == gridDim.x - 1) {
            __hip_atomic_store(a.arrived, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(a.flag, a.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
}

}  // namespace
}  // namespace chx

namespace chx {
namespace {

// Pinned memory comes in slabs of four blocks: an allocation takes 50 us, which every program that sends results to the
// host, and every reader of a small array, would pay.
struct Slab {
    char* pinned = nullptr;
    uint32_t* arrived = nullptr;
    int blocks = 0;  // of it that exist, in use or waiting
};
constexpr int kSlabBlocks = 4;

}  // namespace
}  // namespace chx

struct chx_hip_copyout {
    chx::Slab* slab = nullptr;
    char* pinned = nullptr;  // the results, and behind them the flag
    uint32_t* arrived = nullptr;
    size_t capacity = 0;
    uint32_t seq = 0;
    size_t at[chx::kMaxRanges] = {};
    hipStream_t stream = nullptr;  // of the last enqueue
    bool pending = false;
    int device = 0;
};

namespace chx {
namespace {

std::atomic<uint32_t>* flag_of(const chx_hip_copyout* c) {
    return reinterpret_cast<std::atomic<uint32_t>*>(c->pinned + c->capacity);
}

// Blocks that nobody uses, at most kKept of them.
constexpr size_t kKept = 2 * kSlabBlocks, kBlockBytes = kMostBytes + 16 * kMaxRanges + 64;
std::mutex g_mutex;
std::vector<chx_hip_copyout*> g_free;

// (g_mutex held)
void drop(chx_hip_copyout* c) {
    if (--c->slab->blocks == 0) {
        if (c->slab->arrived) (void)hipFree(c->slab->arrived);
        if (c->slab->pinned) (void)hipHostFree(c->slab->pinned);
        delete c->slab;
    }
    delete c;
}

// Whether a kernel on `device`, the current one, may read p.  Another device's memory, pinned and pageable host memory are
// hipMemcpy's.
bool memory_of(int device, const void* p) {
    hipPointerAttribute_t at;
    if (hipPointerGetAttributes(&at, p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return at.type == hipMemoryTypeDevice && at.device == device;
}

bool stream_of(int device, hipStream_t s) {
    int current = 0;
    if (hipGetDevice(&current) != hipSuccess || current != device) return false;
    if (s == nullptr) return true;
    hipDevice_t of_stream = 0;
    if (hipStreamGetDevice(s, &of_stream) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return of_stream == device;
}

chx_hip_copyout* take(int device) {
    for (size_t i = 0; i < g_free.size(); ++i) {
        if (g_free[i]->device != device) continue;
        chx_hip_copyout* c = g_free[i];
        g_free.erase(g_free.begin() + (long)i);
        return c;
    }
    return nullptr;
}

}  // namespace

// Returns false, with nothing done, when the copy is not one for this path (or no block could be allocated).
bool small_copy_to_host(void* dst, const void* src, size_t bytes, hipStream_t s, int* rc) {
    if (bytes > kMostBytes || stream_is_capturing(s)) return false;
    chx_hip_copyout* c = nullptr;
    if (chx_hip_copyout_create(kMostBytes, &c) != CHX_HIP_OK) return false;
    *rc = chx_hip_copyout_enqueue(c, &src, &bytes, 1, s);
    if (*rc == CHX_HIP_EUNSUPPORTED) {
        chx_hip_copyout_destroy(c);
        return false;
    }
    if (*rc == CHX_HIP_OK) *rc = chx_hip_copyout_wait(c);
    if (*rc == CHX_HIP_OK) memcpy(dst, chx_hip_copyout_data(c, 0), bytes);
    chx_hip_copyout_destroy(c);
    return true;
}

}  // namespace chx

using namespace chx;

extern "C" int chx_hip_copyout_create(size_t bytes, chx_hip_copyout** out) {
    CHX_REQUIRE(out != nullptr, "copyout: null output");
    *out = nullptr;
    if (bytes > kMostBytes) CHX_FAIL(CHX_HIP_EUNSUPPORTED, "copyout: %zu bytes are more than the %zu of this path", bytes, kMostBytes);
    int device = 0;
    CHX_HIP_CALL(hipGetDevice(&device));
    std::lock_guard<std::mutex> lock(g_mutex);
    chx_hip_copyout* c = take(device);
    if (!c) {
        void *p = nullptr, *d = nullptr;
        hipError_t e = hipHostMalloc(&p, kSlabBlocks * (kBlockBytes + 64), hipHostMallocDefault);
        if (e == hipSuccess) e = hipMalloc(&d, kSlabBlocks * 64);
        if (e == hipSuccess) {
            const uint32_t zeros[kSlabBlocks * 16] = {};
            e = hipMemcpy(d, zeros, sizeof(zeros), hipMemcpyHostToDevice);
        }
        if (e != hipSuccess) {
            (void)hipGetLastError();
            if (d) (void)hipFree(d);
            if (p) (void)hipHostFree(p);
            CHX_FAIL(CHX_HIP_ERUNTIME, "copyout: allocation failed: %s", hipGetErrorString(e));
        }
        Slab* slab = new Slab{static_cast<char*>(p), static_cast<uint32_t*>(d), kSlabBlocks};
        for (int i = 0; i < kSlabBlocks; ++i) {
            chx_hip_copyout* b = new chx_hip_copyout();
            b->slab = slab;
            b->capacity = kBlockBytes;
            b->pinned = slab->pinned + i * (kBlockBytes + 64);
            memset(b->pinned + kBlockBytes, 0, 64);
            b->arrived = slab->arrived + 16 * i;
            b->device = device;
            g_free.push_back(b);
        }
        c = take(device);
    }
    *out = c;
    return CHX_HIP_OK;
}

extern "C" int chx_hip_copyout_enqueue(chx_hip_copyout* c, const void* const* src, const size_t* bytes, int32_t n, void* stream) {
    CHX_REQUIRE(c != nullptr && n >= 0 && (n == 0 || (src != nullptr && bytes != nullptr)), "copyout: null argument");
    if (n > kMaxRanges) CHX_FAIL(CHX_HIP_EUNSUPPORTED, "copyout: %d ranges, at most %d", n, kMaxRanges);
    if (!stream_of(c->device, as_stream(stream))) CHX_FAIL(CHX_HIP_EUNSUPPORTED, "copyout: the stream belongs to another device than the block");
    for (int i = 0; i < n; ++i)
        if (bytes[i] && !memory_of(c->device, src[i])) CHX_FAIL(CHX_HIP_EUNSUPPORTED, "copyout: range %d is not memory of the block's device", i);
    if (c->pending) CHX_PROPAGATE(chx_hip_copyout_wait(c));
    CopyOutArgs a;
    memset(&a, 0, sizeof(a));
    size_t at = 0;
    for (int i = 0; i < n; ++i) {
        CHX_REQUIRE(src[i] != nullptr || bytes[i] == 0, "copyout: null source");
        if (bytes[i] > c->capacity || at + bytes[i] > c->capacity) CHX_FAIL(CHX_HIP_EUNSUPPORTED, "copyout: the ranges exceed the block");
        a.src[i] = static_cast<const char*>(src[i]);
        a.bytes[i] = (uint32_t)bytes[i];
        a.at[i] = (uint32_t)at;
        c->at[i] = at;
        at += (bytes[i] + 15) / 16 * 16;
    }
    a.n = n;
    a.dst = c->pinned;
    a.arrived = c->arrived;
    a.flag = reinterpret_cast<uint32_t*>(c->pinned + c->capacity);
    a.seq = ++c->seq;
    c->stream = as_stream(stream);
    // eight work-groups keep the link to the host busy; more only wait for each other's fences
    const unsigned blocks = (unsigned)std::min<size_t>(8, (at + kThreads * 16 - 1) / (kThreads * 16));
    copy_out_kernel<<<blocks ? blocks : 1, kThreads, 0, c->stream>>>(a);
    CHX_PROPAGATE(launch_check("copy_out_kernel"));
    c->pending = true;
    return CHX_HIP_OK;
}

extern "C" int chx_hip_copyout_wait(chx_hip_copyout* c) {
    CHX_REQUIRE(c != nullptr, "copyout: null argument");
    if (!c->pending) return CHX_HIP_OK;
    const auto start = std::chrono::steady_clock::now();
    for (uint32_t spins = 1; flag_of(c)->load(std::memory_order_acquire) != c->seq; ++spins) {
        __builtin_ia32_pause();
        // after a while the runtime waits, which also reports what went wrong on the device
        if (spins % 1024 == 0 && std::chrono::steady_clock::now() - start > std::chrono::milliseconds(2)) {
            CHX_HIP_CALL(hipStreamSynchronize(c->stream));
            CHX_REQUIRE(flag_of(c)->load(std::memory_order_acquire) == c->seq, "copyout: the stream is done, the copy is not");
        }
    }
    c->pending = false;
    return CHX_HIP_OK;
}

extern "C" const void* chx_hip_copyout_data(const chx_hip_copyout* c, int32_t i) {
    return c && i >= 0 && i < kMaxRanges ? c->pinned + c->at[i] : nullptr;
}

extern "C" void chx_hip_copyout_destroy(chx_hip_copyout* c) {
    if (!c) return;
    if (c->pending) (void)hipStreamSynchronize(c->stream);
    c->pending = false;
    std::lock_guard<std::mutex> lock(g_mutex);
    if (g_free.size() < kKept) g_free.push_back(c);
    else drop(c);
}
