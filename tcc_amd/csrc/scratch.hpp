// Device memory of the builders (COO -> BCSR / BCSC / hybrid), kept between
// calls: their scratch and the arrays they hand out.  A hipMalloc / hipFree
// pair costs 30-300 us, as much as a whole build of a sampled subgraph, and
// memory freed is cleared before it is given out again: builds of 57M edges
// in a row (1.5 GB each) took 16.7 ms a build, 6.9 ms with a pause between.
//
// A kept block has no work left that could touch it: scratch comes back only
// after its call has waited for its stream, handed-out arrays after the
// device is idle (hipFree waits for that too).  So any thread and stream can
// take it next.  At most kPoolKeep bytes are kept per device, the blocks kept
// longest freed first; tcc_release_kept_memory and tcc_swtcf_release_plans free
// them all, and so does any allocation of the library that would otherwise fail
// (every one goes through device_malloc, pool_malloc or Scratch).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace tcc {

constexpr std::size_t kPoolKeep = std::size_t(2) << 30;

// At least `bytes` on the current device for arrays handed to the caller;
// pool_free gives them back from any thread.
hipError_t pool_malloc(void** p, std::size_t bytes);
hipError_t pool_free(void* p);

// Frees every kept block of every device.
void pool_release();

// hipMalloc that frees the kept blocks and tries again where memory is short;
// hipFree frees its result.
hipError_t device_malloc(void** p, std::size_t bytes);
template <typename T>
hipError_t device_malloc(T** p, std::size_t bytes) {
    return device_malloc(reinterpret_cast<void**>(p), bytes);
}

// One call's scratch, with a small host-mapped mailbox that its kernels
// write and the host reads after a wait.
class Scratch {
public:
    Scratch() = default;
    Scratch(const Scratch&) = delete;
    Scratch& operator=(const Scratch&) = delete;
    ~Scratch();

    // At least `bytes` on the current device for work on `st`.
    hipError_t take(std::size_t bytes, hipStream_t st);
    hipError_t wait() { return hipStreamSynchronize(st_); }
    // wait() after the call's last work: nothing may be queued after it.
    hipError_t finish();
    // The call has waited for the stream elsewhere and queues nothing more.
    void idle() { busy_ = false; }

    char* data() const { return p_; }
    std::uint32_t* mail() const { return mailDev_; }  // [16] words, their device address
    std::uint32_t* mailHost() const { return mailHost_; }
    const volatile std::uint32_t* read() const { return mailHost_; }

private:
    char* p_ = nullptr;
    std::size_t bytes_ = 0;
    std::uint32_t* mailHost_ = nullptr;
    std::uint32_t* mailDev_ = nullptr;
    hipStream_t st_ = nullptr;
    int dev_ = 0;
    bool busy_ = false;  // work may be queued: taken and not finished
};

}  // namespace tcc
