#include "device_cache.h"

namespace chainer_compiler {
namespace runtime {

namespace {

// 512-byte steps, and above 64 KB steps of an eighth of the power of two below: at most 12.5 % of a block is unused
size_t SizeClass(size_t bytes) {
    size_t step = 512;
    while (step * 128 < bytes) step *= 2;
    return (bytes + step - 1) / step * step;
}

}  // namespace

DeviceCache& DeviceCache::Get() {
    static DeviceCache* cache = new DeviceCache();  // outlives every array: never destroyed
    return *cache;
}

std::shared_ptr<void> DeviceCache::Allocate(size_t bytes) {
    const size_t size = SizeClass(bytes);
    void* p = nullptr;
    {
        std::lock_guard<std::mutex> lock(mu_);
        auto it = free_.find(size);
        if (it != free_.end() && !it->second.empty()) {
            p = it->second.back();
            it->second.pop_back();
            cached_ -= size;
        }
    }
    if (!p && chx_hip_malloc(&p, size) != 0) {
        Trim();  // what is kept may be what is missing
        CHXVM_HIP_CALL(chx_hip_malloc(&p, size));
    }
    return std::shared_ptr<void>(p, [this, size](void* q) { Release(q, size); });
}

void DeviceCache::Release(void* p, size_t size) {
    {
        std::lock_guard<std::mutex> lock(mu_);
        if (programs_ > 0 && size <= kLargestKept && cached_ + size <= kMostCached) {
            free_[size].push_back(p);
            cached_ += size;
            return;
        }
    }
    (void)chx_hip_free(p);
}

void DeviceCache::Trim() {
    std::map<size_t, std::vector<void*>> blocks;
    {
        std::lock_guard<std::mutex> lock(mu_);
        blocks.swap(free_);
        cached_ = 0;
    }
    for (auto& c : blocks)
        for (void* p : c.second) (void)chx_hip_free(p);
}

void DeviceCache::AddProgram() {
    std::lock_guard<std::mutex> lock(mu_);
    ++programs_;
}

void DeviceCache::RemoveProgram() {
    bool last = false;
    {
        std::lock_guard<std::mutex> lock(mu_);
        last = --programs_ == 0;
    }
    if (last) Trim();
}

}  // namespace runtime
}  // namespace chainer_compiler

chainerx::DeviceAllocator& chainerx::DefaultDeviceAllocator() {
    return chainer_compiler::runtime::DeviceCache::Get();
}
