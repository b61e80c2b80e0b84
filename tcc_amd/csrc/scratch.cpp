// The kept device memory of scratch.hpp.
#include "scratch.hpp"

#include <mutex>

namespace tcc {
namespace {

struct Block {
    char* p;
    std::size_t bytes;
    int dev;
};

struct Mail {
    std::uint32_t *host, *dev;
};

// Kept blocks (oldest first), the handed-out arrays whose sizes are known,
// and free mailboxes; fixed tables, so that no path here can throw.  A block
// or mailbox that finds no place is freed, an array that finds none is freed
// when it comes back.  Nothing is freed at exit: the runtime may be gone.
constexpr int kMaxKept = 64, kMaxOut = 256, kMaxMail = 16;
std::mutex g_mutex;
Block g_kept[kMaxKept];
int g_numKept = 0;
Block g_out[kMaxOut];
int g_numOut = 0;
Mail g_mail[kMaxMail];
int g_numMail = 0;

// A kept block of at least `bytes` and at most `most` of the device (the
// smallest such), taken out; bytes = 0 for none.  Under the lock.
Block take_kept(std::size_t bytes, std::size_t most, int dev) {
    int best = -1;
    for (int i = 0; i < g_numKept; ++i)
        if (g_kept[i].dev == dev && g_kept[i].bytes >= bytes && g_kept[i].bytes <= most &&
            (best < 0 || g_kept[i].bytes < g_kept[best].bytes))
            best = i;
    if (best < 0) return Block{nullptr, 0, dev};
    const Block b = g_kept[best];
    for (int i = best; i + 1 < g_numKept; ++i) g_kept[i] = g_kept[i + 1];
    --g_numKept;
    return b;
}

// Keeps an idle block, the oldest of its device making room.  Under the lock.
void keep(const Block& b) {
    if (b.bytes > kPoolKeep) {
        (void)hipFree(b.p);
        return;
    }
    std::size_t kept = b.bytes;
    for (int i = 0; i < g_numKept; ++i)
        if (g_kept[i].dev == b.dev) kept += g_kept[i].bytes;
    for (int i = 0; i < g_numKept && (kept > kPoolKeep || g_numKept == kMaxKept);) {
        if (g_kept[i].dev != b.dev) {
            ++i;
            continue;
        }
        kept -= g_kept[i].bytes;
        (void)hipFree(g_kept[i].p);
        for (int j = i; j + 1 < g_numKept; ++j) g_kept[j] = g_kept[j + 1];
        --g_numKept;
    }
    if (g_numKept < kMaxKept) g_kept[g_numKept++] = b;
    else (void)hipFree(b.p);
}

}  // namespace

hipError_t device_malloc(void** p, std::size_t bytes) {
    hipError_t e = hipMalloc(p, bytes);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        pool_release();
        e = hipMalloc(p, bytes);
    }
    if (e != hipSuccess) *p = nullptr;
    return e;
}

void pool_release() {
    std::lock_guard<std::mutex> lock(g_mutex);
    while (g_numKept > 0) (void)hipFree(g_kept[--g_numKept].p);
}

hipError_t pool_malloc(void** p, std::size_t bytes) {
    *p = nullptr;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    Block b;
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        b = take_kept(bytes, bytes + bytes / 8 + 65536, dev);  // arrays may be held for long: a close fit
    }
    if (!b.p) {
        e = device_malloc(&b.p, bytes);
        if (e != hipSuccess) return e;
        b.bytes = bytes;
    }
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        if (g_numOut < kMaxOut) g_out[g_numOut++] = b;
    }
    *p = b.p;
    return hipSuccess;
}

hipError_t pool_free(void* p) {
    if (!p) return hipSuccess;
    Block b{nullptr, 0, 0};
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        for (int i = 0; i < g_numOut; ++i)
            if (g_out[i].p == p) {
                b = g_out[i];
                g_out[i] = g_out[--g_numOut];
                break;
            }
    }
    int dev = 0;
    if (!b.p || b.bytes > kPoolKeep || hipGetDevice(&dev) != hipSuccess || dev != b.dev) return hipFree(p);
    const hipError_t e = hipDeviceSynchronize();  // as hipFree: work of any stream may read the arrays
    if (e != hipSuccess) return hipFree(p);
    std::lock_guard<std::mutex> lock(g_mutex);
    keep(b);
    return hipSuccess;
}

hipError_t Scratch::take(std::size_t bytes, hipStream_t st) {
    hipError_t e = hipGetDevice(&dev_);
    if (e != hipSuccess) return e;
    st_ = st;
    Block b;
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        b = take_kept(bytes, 4 * bytes + (std::size_t(64) << 20), dev_);  // back at the call's end: any fair fit
        if (g_numMail > 0) {
            mailHost_ = g_mail[--g_numMail].host;
            mailDev_ = g_mail[g_numMail].dev;
        }
    }
    if (!mailHost_) {
        e = hipHostMalloc(reinterpret_cast<void**>(&mailHost_), 64, hipHostMallocMapped | hipHostMallocPortable);
        if (e != hipSuccess) mailHost_ = nullptr;
        if (e == hipSuccess) e = hipHostGetDevicePointer(reinterpret_cast<void**>(&mailDev_), mailHost_, 0);
    }
    if (e == hipSuccess && !b.p) {
        // room for somewhat larger calls to come, where there is room
        b.bytes = bytes + (bytes < kPoolKeep / 8 ? bytes / 4 : 0);
        e = hipMalloc(reinterpret_cast<void**>(&b.p), b.bytes);
        if (e == hipErrorOutOfMemory) {
            (void)hipGetLastError();
            b.bytes = bytes;
            e = device_malloc(&b.p, bytes);
        }
        if (e != hipSuccess) b.p = nullptr;
    }
    p_ = b.p;
    bytes_ = b.bytes;
    busy_ = e == hipSuccess;
    return e;
}

hipError_t Scratch::finish() {
    const hipError_t e = hipStreamSynchronize(st_);
    if (e == hipSuccess) busy_ = false;
    return e;
}

Scratch::~Scratch() {
    const bool reuse = !busy_ || hipStreamSynchronize(st_) == hipSuccess;  // else an error is pending
    std::lock_guard<std::mutex> lock(g_mutex);
    if (p_) {
        if (reuse) keep(Block{p_, bytes_, dev_});
        else (void)hipFree(p_);
    }
    if (mailHost_) {
        if (reuse && mailDev_ && g_numMail < kMaxMail) g_mail[g_numMail++] = Mail{mailHost_, mailDev_};
        else (void)hipHostFree(mailHost_);
    }
}

}  // namespace tcc
