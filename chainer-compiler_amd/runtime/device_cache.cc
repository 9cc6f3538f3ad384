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

int32_t CurrentDevice() {
    int32_t device = 0;
    CHXVM_HIP_CALL(chx_hip_get_device(&device));
    return device;
}

}  // namespace

DeviceCache& DeviceCache::Get() {
    static DeviceCache* cache = new DeviceCache();  // outlives every array: never destroyed
    return *cache;
}

std::shared_ptr<void> DeviceCache::Allocate(size_t bytes) {
    const size_t size = SizeClass(bytes);
    const int32_t device = CurrentDevice();
    void* p = nullptr;
    {
        std::lock_guard<std::mutex> lock(mu_);
        auto it = free_.find({device, size});
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
    return std::shared_ptr<void>(p, [this, size, device](void* q) { Release(q, size, device); });
}

void DeviceCache::Release(void* p, size_t size, int32_t device) {
    // (what is given up while another device is current goes back to the device runtime: the owner has waited for that
    // other device, hipFree waits for this one)
    int32_t current = -1;
    (void)chx_hip_get_device(&current);
    {
        std::lock_guard<std::mutex> lock(mu_);
        if (device == current && programs_ > 0 && size <= kLargestKept && cached_ + size <= kMostCached) {
            free_[{device, size}].push_back(p);
            cached_ += size;
            return;
        }
    }
    (void)chx_hip_free(p);
}

void DeviceCache::Trim() {
    std::map<std::pair<int32_t, size_t>, std::vector<void*>> blocks;
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
