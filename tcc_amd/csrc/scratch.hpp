// Device scratch of the synchronous builders (COO -> BCSR / BCSC), kept
// between calls: a hipMalloc / hipFree pair costs 30-300 us, as much as a
// whole build of a sampled subgraph.  A block belongs to one call at a time
// and is given back only after that call has waited for its stream, so calls
// from any thread and stream can take it next.  At most kScratchKeep bytes
// are kept per device (larger blocks are freed at once); tcc_swtcf_release_plans
// frees them, and so does an allocation that would otherwise fail.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace tcc {

constexpr std::size_t kScratchKeep = 256u << 20;

// One call's scratch, with a small host-mapped mailbox that its kernels
// write and the host reads after finish().
class Scratch {
public:
    Scratch() = default;
    Scratch(const Scratch&) = delete;
    Scratch& operator=(const Scratch&) = delete;
    ~Scratch();

    // At least `bytes` on the current device for work on `st`.
    hipError_t take(std::size_t bytes, hipStream_t st);
    // Waits for the stream; the mailbox then holds what the kernels wrote.
    // finish() is for the call's last work: nothing may be queued after it.
    hipError_t wait() { return hipStreamSynchronize(st_); }
    hipError_t finish();

    char* data() const { return p_; }
    std::uint32_t* mail() const { return mailDev_; }               // [16] words, their device address
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

// Frees every kept block of every device.
void release_scratch();

// hipMalloc; on failure once more after the kept blocks are freed.
hipError_t malloc_or_release(void** p, std::size_t bytes);

}  // namespace tcc
