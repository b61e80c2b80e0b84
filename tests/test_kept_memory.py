"""The builders' kept device memory (csrc/scratch.cpp) over a stand-in for the
HIP runtime with a fixed amount of memory, no GPU: what is kept never makes
another allocation of the library fail, never exceeds its bound, and is handed
out once at a time, with several threads too."""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "tcc_amd", "csrc")

PROGRAM = r"""
#include "scratch.hpp"

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <mutex>
#include <thread>
#include <vector>

// device memory: addresses from a counter, sizes in a map
static std::mutex mu;
static std::map<char*, std::size_t> blocks;
static std::size_t used = 0, capacity = 0;
static char* next_address = reinterpret_cast<char*>(1ull << 40);
static thread_local int device = 0;

extern "C" {
hipError_t hipGetDevice(int* d) { *d = device; return hipSuccess; }
hipError_t hipMalloc(void** p, std::size_t n) {
    std::lock_guard<std::mutex> lock(mu);
    if (used + n > capacity) return hipErrorOutOfMemory;
    used += n;
    *p = next_address;
    blocks[next_address] = n;
    next_address += n + 4096;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    std::lock_guard<std::mutex> lock(mu);
    auto it = blocks.find(static_cast<char*>(p));
    if (it == blocks.end()) { std::printf("freed twice\n"); std::abort(); }
    used -= it->second;
    blocks.erase(it);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, std::size_t n, unsigned) { *p = std::calloc(1, n); return hipSuccess; }
hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) { *d = h; return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
}

#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)

constexpr std::size_t MiB = 1 << 20, GiB = 1 << 30;

static int one_thread() {
    capacity = 5 * GiB;
    { tcc::Scratch s; CHECK(s.take(3 * GiB / 2, nullptr) == hipSuccess); CHECK(s.finish() == hipSuccess); }
    CHECK(used >= 3 * GiB / 2 && used <= tcc::kPoolKeep);  // kept
    void* p = nullptr;
    CHECK(tcc::device_malloc(&p, 4 * GiB) == hipSuccess);  // not before what is kept is freed
    CHECK(hipFree(p) == hipSuccess);
    CHECK(tcc::device_malloc(&p, 6 * GiB) == hipErrorOutOfMemory && p == nullptr);
    CHECK(used == 0);
    // handed-out arrays: kept, taken again by a close fit, given back to others
    CHECK(tcc::pool_malloc(&p, GiB) == hipSuccess && tcc::pool_free(p) == hipSuccess && used == GiB);
    void* q = nullptr;
    CHECK(tcc::pool_malloc(&q, GiB - 100) == hipSuccess && q == p && tcc::pool_free(q) == hipSuccess);
    CHECK(tcc::pool_malloc(&q, 9 * GiB / 2) == hipSuccess && tcc::pool_free(q) == hipSuccess && used == 0);
    // a scratch that fits without the room for larger ones
    capacity = 220 * MiB;
    { tcc::Scratch s; CHECK(s.take(200 * MiB, nullptr) == hipSuccess); CHECK(s.finish() == hipSuccess); }
    tcc::pool_release();
    CHECK(used == 0);
    // never more than the bound, whatever is released
    capacity = 64 * GiB;
    std::vector<void*> all;
    for (int i = 0; i < 300; ++i) {
        void* x = nullptr;
        CHECK(tcc::pool_malloc(&x, (i % 7 + 1) * 20 * MiB) == hipSuccess);
        all.push_back(x);
    }
    for (void* x : all) CHECK(tcc::pool_free(x) == hipSuccess);
    CHECK(used <= tcc::kPoolKeep);
    tcc::pool_release();
    CHECK(used == 0 && blocks.empty());
    return 0;
}

static std::atomic<int> bad{0};
static std::mutex owned_mu;
static std::map<char*, std::size_t> owned;  // ranges in use

static void own(char* p, std::size_t n) {
    std::lock_guard<std::mutex> lock(owned_mu);
    auto it = owned.lower_bound(p);
    if (it != owned.end() && it->first < p + n) ++bad;
    if (it != owned.begin() && std::prev(it)->first + std::prev(it)->second > p) ++bad;
    owned[p] = n;
}
static void disown(char* p) {
    std::lock_guard<std::mutex> lock(owned_mu);
    owned.erase(p);
}

static void worker(unsigned seed) {
    device = static_cast<int>(seed % 2);
    unsigned x = seed * 2654435761u + 1;
    auto rnd = [&] { x = x * 1664525u + 1013904223u; return x >> 8; };
    std::vector<void*> mine;
    for (int i = 0; i < 4000; ++i) {
        const std::size_t n = (rnd() % 64 + 1) * MiB + rnd() % 1000;
        if (rnd() % 2) {
            tcc::Scratch s;
            if (s.take(n, nullptr) != hipSuccess) continue;
            own(s.data(), n);
            if (rnd() % 4 == 0) std::this_thread::yield();
            disown(s.data());
            if (rnd() % 2) (void)s.finish();
        } else if (mine.size() < 8 && rnd() % 3) {
            void* p = nullptr;
            if (tcc::pool_malloc(&p, n) != hipSuccess) continue;
            own(static_cast<char*>(p), n);
            mine.push_back(p);
        } else if (!mine.empty()) {
            disown(static_cast<char*>(mine.back()));
            if (tcc::pool_free(mine.back()) != hipSuccess) ++bad;
            mine.pop_back();
        }
        if (rnd() % 500 == 0) tcc::pool_release();
    }
    for (void* p : mine) {
        disown(static_cast<char*>(p));
        (void)tcc::pool_free(p);
    }
}

int main() {
    if (one_thread()) return 1;
    capacity = 6 * GiB;  // short at times
    std::vector<std::thread> threads;
    for (unsigned t = 0; t < 8; ++t) threads.emplace_back(worker, t);
    for (auto& t : threads) t.join();
    CHECK(bad == 0);
    CHECK(used <= 2 * tcc::kPoolKeep);  // two devices
    tcc::pool_release();
    CHECK(used == 0 && blocks.empty());
    std::printf("OK\n");
    return 0;
}
"""


def test_kept_memory_never_stands_in_the_way(tmp_path):
    src, exe = tmp_path / "kept.cpp", tmp_path / "kept"
    src.write_text(PROGRAM)
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-pthread",
                        "-D__HIP_PLATFORM_AMD__=1", "-I/opt/rocm/include", f"-I{CSRC}", str(src),
                        os.path.join(CSRC, "scratch.cpp"), "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "OK" in r.stdout, r.stdout + r.stderr


def test_every_allocation_can_take_what_is_kept():
    """No device allocation of the library but scratch.cpp's own asks the
    runtime directly."""
    for name in sorted(os.listdir(CSRC)):
        if name.startswith("scratch.") or not name.endswith((".hip", ".hpp", ".cpp")):
            continue
        text = re.sub(r"//[^\n]*", "", open(os.path.join(CSRC, name)).read())
        calls = re.findall(r"\bhipMalloc\w*\s*\(", text)
        # the extension's device_malloc: the runtime, then what is kept, then again
        assert len(calls) == (2 if name == "spmm_cnic_ext.cpp" else 0), (name, calls)
