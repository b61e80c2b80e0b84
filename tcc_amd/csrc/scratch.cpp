// The kept scratch blocks of scratch.hpp.
#include "scratch.hpp"

#include <mutex>

namespace tcc {
namespace {

struct Block {
    char* p;
    std::size_t bytes;
    std::uint32_t* mailHost;
    std::uint32_t* mailDev;
    int dev;
};

// The kept blocks, all devices (not freed at exit: the runtime may be gone).
constexpr int kMaxBlocks = 32;
std::mutex g_mutex;
Block g_kept[kMaxBlocks];
int g_count = 0;

void free_block(const Block& b) {
    (void)hipFree(b.p);
    (void)hipHostFree(b.mailHost);
}

}  // namespace

void release_scratch() {
    std::lock_guard<std::mutex> lock(g_mutex);
    while (g_count > 0) free_block(g_kept[--g_count]);
}

hipError_t malloc_or_release(void** p, std::size_t bytes) {
    hipError_t e = hipMalloc(p, bytes);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        release_scratch();
        e = hipMalloc(p, bytes);
    }
    return e;
}

hipError_t Scratch::take(std::size_t bytes, hipStream_t st) {
    hipError_t e = hipGetDevice(&dev_);
    if (e != hipSuccess) return e;
    st_ = st;
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        int best = -1;
        for (int i = 0; i < g_count; ++i)
            if (g_kept[i].dev == dev_ && g_kept[i].bytes >= bytes && (best < 0 || g_kept[i].bytes < g_kept[best].bytes))
                best = i;
        if (best >= 0) {
            const Block b = g_kept[best];
            g_kept[best] = g_kept[--g_count];
            p_ = b.p;
            bytes_ = b.bytes;
            mailHost_ = b.mailHost;
            mailDev_ = b.mailDev;
        }
    }
    if (!p_) {
        // a kept block gets room for somewhat larger calls to come
        const std::size_t want = bytes + (bytes < kScratchKeep / 2 ? bytes / 4 : 0);
        e = malloc_or_release(reinterpret_cast<void**>(&p_), want);
        if (e != hipSuccess) {
            p_ = nullptr;
            return e;
        }
        bytes_ = want;
        e = hipHostMalloc(reinterpret_cast<void**>(&mailHost_), 64, hipHostMallocMapped);
        if (e != hipSuccess) mailHost_ = nullptr;
        if (e == hipSuccess) e = hipHostGetDevicePointer(reinterpret_cast<void**>(&mailDev_), mailHost_, 0);
        if (e != hipSuccess) {
            (void)hipFree(p_);
            if (mailHost_) (void)hipHostFree(mailHost_);
            p_ = nullptr;
            mailHost_ = nullptr;
            return e;
        }
    }
    busy_ = true;
    return hipSuccess;
}

hipError_t Scratch::finish() {
    const hipError_t e = hipStreamSynchronize(st_);
    if (e == hipSuccess) busy_ = false;
    return e;
}

Scratch::~Scratch() {
    if (!p_) return;
    const Block b{p_, bytes_, mailHost_, mailDev_, dev_};
    if (busy_ && hipStreamSynchronize(st_) != hipSuccess) {
        free_block(b);  // an error is pending: nothing of this call is used again
        return;
    }
    if (bytes_ <= kScratchKeep) {
        std::lock_guard<std::mutex> lock(g_mutex);
        std::size_t kept = 0;
        for (int i = 0; i < g_count; ++i)
            if (g_kept[i].dev == dev_) kept += g_kept[i].bytes;
        // a larger block serves every smaller call: smaller ones make room
        for (int i = 0; i < g_count && kept + bytes_ > kScratchKeep;) {
            if (g_kept[i].dev == dev_ && g_kept[i].bytes < bytes_) {
                kept -= g_kept[i].bytes;
                free_block(g_kept[i]);
                g_kept[i] = g_kept[--g_count];
            } else {
                ++i;
            }
        }
        if (kept + bytes_ <= kScratchKeep && g_count < kMaxBlocks) {
            g_kept[g_count++] = b;
            return;
        }
    }
    free_block(b);
}

}  // namespace tcc
