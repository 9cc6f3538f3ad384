// A device runtime without a device, for tests of the host side: loaded before libchx_hip.so (RTLD_GLOBAL), its functions
// take the place of libamdhip64's.  Two devices, whose memory is host memory; streams, captures and graphs as far as the
// library uses them; kernels are written to a log instead of run, all but the one that copies results to the host.
//   hh_log / hh_clear         what happened since hh_clear, a line each
//   hh_device_of(p)           the device whose memory p is, -1: none
//   hh_prefer(text)           event pairs around launches of kernels with this in their name measure a tenth of the others
//   hh_no_memory(n)           there is none for requests of exactly n bytes (0: for all)
//   hh_hold(1), hh_held(), hh_release()
//                             copies to the host stay queued, and the first caller of hipStreamSynchronize stays in it,
//                             until the release; later callers let all queued copies happen, as a device would
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>

#include <cxxabi.h>

#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace {

struct Block {
    size_t size;
    int device;  // -1: host
};
struct CopyOut {  // the argument block of copy_out_kernel (csrc/copyout.hip)
    const char* src[8];
    uint32_t bytes[8], at[8];
    int32_t n;
    char* dst;
    uint32_t* arrived;
    uint32_t* flag;
    uint32_t seq;
};
struct Stream {
    int device;
    bool capturing = false, broken = false;
};
struct Event {
    int preferred = 0;
};

// (never destroyed: the library unregisters its code objects when the process ends)
std::recursive_mutex& g_mutex = *new std::recursive_mutex;
std::condition_variable_any& g_changed = *new std::condition_variable_any;
std::map<char*, Block>& g_blocks = *new std::map<char*, Block>;
std::map<const void*, std::string>& g_kernels = *new std::map<const void*, std::string>;
std::map<hipStream_t, Stream>& g_streams = *new std::map<hipStream_t, Stream>;
std::vector<CopyOut>& g_queued = *new std::vector<CopyOut>;
std::string& g_log = *new std::string;
std::string& g_prefer = *new std::string;
bool g_hold = false;
int g_held = 0;
int g_preferred_launches = 0;
size_t g_no_memory = 0;
thread_local int t_device = 0;
thread_local dim3 t_grid, t_block;
thread_local size_t t_lds;
thread_local hipStream_t t_stream;
thread_local hipError_t t_error = hipSuccess;

typedef std::lock_guard<std::recursive_mutex> Lock;

void note(const std::string& line) {
    Lock lock(g_mutex);
    g_log += line + "\n";
}

hipError_t allocate(void** p, size_t n, int device) {
    Lock lock(g_mutex);
    if (n != 0 && n == g_no_memory) return t_error = hipErrorOutOfMemory;
    char* q = static_cast<char*>(calloc(1, n ? n : 1));
    if (!q) return hipErrorOutOfMemory;
    g_blocks[q] = Block{n, device};
    *p = q;
    return hipSuccess;
}

hipError_t release(void* p) {
    Lock lock(g_mutex);
    if (!p) return hipSuccess;
    auto it = g_blocks.find(static_cast<char*>(p));
    if (it == g_blocks.end()) return hipErrorInvalidValue;
    free(it->first);
    g_blocks.erase(it);
    return hipSuccess;
}

// -2: not memory of this runtime
int device_of(const void* p) {
    Lock lock(g_mutex);
    auto it = g_blocks.upper_bound(const_cast<char*>(static_cast<const char*>(p)));
    if (it == g_blocks.begin()) return -2;
    --it;
    return static_cast<const char*>(p) < it->first + (it->second.size ? it->second.size : 1) ? it->second.device : -2;
}

bool recording(hipStream_t s) {
    auto it = g_streams.find(s);
    return it != g_streams.end() && it->second.capturing;
}

void deliver(const CopyOut& c) {
    for (int i = 0; i < c.n; ++i) memcpy(c.dst + c.at[i], c.src[i], c.bytes[i]);
    __atomic_store_n(c.flag, c.seq, __ATOMIC_RELEASE);
}

void deliver_queued() {
    Lock lock(g_mutex);
    for (const CopyOut& c : g_queued) deliver(c);
    g_queued.clear();
}

hipError_t stop(hipStream_t s) {  // a call that a recording stream does not take
    g_streams[s].broken = true;
    note("refused while recording");
    return hipErrorStreamCaptureUnsupported;
}

}  // namespace

extern "C" {

const char* hh_log() {
    static std::string copy;
    Lock lock(g_mutex);
    copy = g_log;
    return copy.c_str();
}
void hh_clear() {
    Lock lock(g_mutex);
    g_log.clear();
}
int hh_device_of(const void* p) {
    return device_of(p);
}
void hh_prefer(const char* text) {
    Lock lock(g_mutex);
    g_prefer = text;
}
void hh_no_memory(size_t n) {
    Lock lock(g_mutex);
    g_no_memory = n;
}
void hh_hold(int on) {
    Lock lock(g_mutex);
    g_hold = on != 0;
    g_held = 0;
}
int hh_held() {
    Lock lock(g_mutex);
    return g_held;
}
void hh_release() {
    Lock lock(g_mutex);
    g_hold = false;
    deliver_queued();
    g_changed.notify_all();
}

void** __hipRegisterFatBinary(const void*) {
    static void* none = nullptr;
    return &none;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    Lock lock(g_mutex);
    int status = 0;
    char* d = abi::__cxa_demangle(name, nullptr, nullptr, &status);
    g_kernels[host] = d ? d : name;
    free(d);
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t s) {
    t_grid = grid;
    t_block = block;
    t_lds = lds;
    t_stream = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* s) {
    *grid = t_grid;
    *block = t_block;
    *lds = t_lds;
    *s = t_stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void** args, size_t lds, hipStream_t s) {
    Lock lock(g_mutex);
    const std::string& name = g_kernels[f];
    char line[160];
    snprintf(line, sizeof(line), " grid=%u,%u,%u block=%u lds=%zu stream=%p device=%d", grid.x, grid.y, grid.z, block.x, lds, (void*)s, t_device);
    note("launch " + name + line);
    if (!g_prefer.empty() && name.find(g_prefer) != std::string::npos) ++g_preferred_launches;
    if (name.find("copy_out_kernel") != std::string::npos && !recording(s)) {
        CopyOut c;
        memcpy(&c, args[0], sizeof(c));
        if (g_hold) g_queued.push_back(c);
        else deliver(c);
    }
    return hipSuccess;
}

hipError_t hipGetDeviceCount(int* n) {
    *n = 2;
    return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
    *d = t_device;
    return hipSuccess;
}
hipError_t hipSetDevice(int d) {
    t_device = d;
    return hipSuccess;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {  // (a macro: the current version of the struct)
    memset(p, 0, sizeof(*p));
    strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t) {
    return "an error of the stand-in device runtime";
}
hipError_t hipGetLastError() {
    const hipError_t e = t_error;
    t_error = hipSuccess;
    return e;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
    return allocate(p, 1 << 16, t_device);
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) {
    return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
    *n = 2;
    return hipSuccess;
}

hipError_t hipMalloc(void** p, size_t n) {
    note("hipMalloc " + std::to_string(n));
    return allocate(p, n, t_device);
}
hipError_t hipFree(void* p) {
    note("hipFree");
    return release(p);
}
hipError_t hipMallocAsync(void** p, size_t n, hipStream_t s) {
    if (recording(s)) return stop(s);
    const hipError_t e = allocate(p, n, t_device);
    char line[96];
    snprintf(line, sizeof(line), "hipMallocAsync %zu stream=%p", n, (void*)s);
    note(line);
    return e;
}
hipError_t hipFreeAsync(void* p, hipStream_t) {
    return release(p);
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    return allocate(p, n, -1);
}
hipError_t hipHostFree(void* p) {
    return release(p);
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
    memset(a, 0, sizeof(*a));
    const int d = device_of(p);
    if (d == -2) return hipErrorInvalidValue;
    a->type = d < 0 ? hipMemoryTypeHost : hipMemoryTypeDevice;
    a->device = d < 0 ? 0 : d;
    return hipSuccess;
}
hipError_t hipMemcpy(void* dst, const void* src, size_t n, hipMemcpyKind) {
    memcpy(dst, src, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind, hipStream_t) {
    note("hipMemcpyAsync " + std::to_string(n));
    memcpy(dst, src, n);
    return hipSuccess;
}
hipError_t hipMemcpy2DAsync(void* dst, size_t dp, const void* src, size_t sp, size_t w, size_t h, hipMemcpyKind, hipStream_t) {
    for (size_t i = 0; i < h; ++i) memcpy(static_cast<char*>(dst) + i * dp, static_cast<const char*>(src) + i * sp, w);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t) {
    memset(p, v, n);
    return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    Lock lock(g_mutex);
    *s = reinterpret_cast<hipStream_t>(malloc(64));
    g_streams[*s] = Stream{t_device};
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    Lock lock(g_mutex);
    g_streams.erase(s);
    return hipSuccess;
}
hipError_t hipStreamGetDevice(hipStream_t s, hipDevice_t* d) {
    Lock lock(g_mutex);
    *d = g_streams.count(s) ? g_streams[s].device : t_device;
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
    std::unique_lock<std::recursive_mutex> lock(g_mutex);
    if (recording(s)) return stop(s);
    note("hipStreamSynchronize");
    if (g_hold && g_held++ == 0) {
        g_changed.wait(lock, [] { return !g_hold; });
        return hipSuccess;
    }
    deliver_queued();
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() {
    note("hipDeviceSynchronize device=" + std::to_string(t_device));
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) {
    Lock lock(g_mutex);
    g_streams[s].capturing = true;
    g_streams[s].broken = false;
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* st) {
    Lock lock(g_mutex);
    *st = recording(s) ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t* g) {
    Lock lock(g_mutex);
    g_streams[s].capturing = false;
    *g = reinterpret_cast<hipGraph_t>(&g_log);
    return g_streams[s].broken ? hipErrorStreamCaptureInvalidated : hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    *e = reinterpret_cast<hipGraphExec_t>(&g_log);
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) {
    return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t) {
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) {
    note("hipGraphLaunch");
    return hipSuccess;
}

hipError_t hipEventCreate(hipEvent_t* e) {
    *e = reinterpret_cast<hipEvent_t>(new Event);
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    delete reinterpret_cast<Event*>(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
    Lock lock(g_mutex);
    reinterpret_cast<Event*>(e)->preferred = g_preferred_launches;
    return hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b) {
    *ms = reinterpret_cast<Event*>(b)->preferred > reinterpret_cast<Event*>(a)->preferred ? 0.1f : 1.0f;
    return hipSuccess;
}

hipError_t hipModuleLoadData(hipModule_t* m, const void*) {
    note("hipModuleLoadData");
    *m = reinterpret_cast<hipModule_t>(&g_log);
    return hipSuccess;
}
hipError_t hipModuleGetFunction(hipFunction_t* f, hipModule_t, const char* name) {
    *f = reinterpret_cast<hipFunction_t>(strdup(name));
    return hipSuccess;
}
hipError_t hipModuleLaunchKernel(hipFunction_t f, unsigned gx, unsigned, unsigned, unsigned, unsigned, unsigned, unsigned, hipStream_t, void**, void**) {
    note("launch " + std::string(reinterpret_cast<const char*>(f)) + " grid=" + std::to_string(gx));
    return hipSuccess;
}

}  // extern "C"
