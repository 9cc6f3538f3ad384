// Device memory of eager runs.  hipFree waits for all work on the device: a run that frees every value after its last
// reader (as programs do) stopped the host after each instruction, 60 times in a ResNet-50, and the device idled while
// the host caught up (2.3 ms for a batch of 8 whose kernels take 0.4).  Blocks released by one value are kept for the
// next request of their size class on the same device instead.
//
// All users are eager runs, whose work goes to the null stream: a block handed out again is written only behind the work
// that still reads it.  Memory that leaves a run (outputs, a program's constants) comes back after the device has been
// synchronized (chxvm_outputs_destroy, chxvm_program_destroy), as hipFree did it.
#pragma once

#include <map>
#include <mutex>
#include <utility>
#include <vector>

#include "chainerx_lite.h"

namespace chainer_compiler {
namespace runtime {

class DeviceCache : public chainerx::DeviceAllocator {
public:
    static DeviceCache& Get();  // the process's one

    std::shared_ptr<void> Allocate(size_t bytes) override;
    // Everything that is not in use goes back to the device runtime (also when the last program is destroyed).
    void Trim();
    void AddProgram();
    void RemoveProgram();

private:
    DeviceCache() = default;
    void Release(void* p, size_t size, int32_t device);

    static constexpr size_t kMostCached = size_t(1) << 30;    // bytes kept beyond those in use
    static constexpr size_t kLargestKept = size_t(256) << 20;  // larger blocks are not kept

    std::mutex mu_;
    std::map<std::pair<int32_t, size_t>, std::vector<void*>> free_;  // by device and size class
    size_t cached_ = 0;
    int64_t programs_ = 0;
};

}  // namespace runtime
}  // namespace chainer_compiler
