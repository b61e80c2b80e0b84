// COO -> BCSR / BCSC construction on gfx950.
//
// The reference's producer of these arrays (ipc_service, outside the
// repository) is absent; the layout here is the one its kernels consume
// (spmm_cnic/src/core/spmm_kernel.cu:87-121 for BCSR, :521-524, :600-615 and
// :689-690 for BCSC, :88-101 for the value order):
//   BCSR: per 8-row window, its distinct columns ascending, 8 per block.
//   BCSC: per 8-source window, its destination rows ordered by (degree desc,
//         dst asc), 8 per block.
// Both are one build: edges (a, b) are grouped by window a / 8 (a = row for
// BCSR, source for BCSC), and each window needs the list of its distinct b,
// ascending, with the 8-bit mask of the a % 8 that have it.
//   1. Grouping.  A COO whose windows never decrease (listed row by row, as
//      CSR gives it, for BCSR) is used in place: one pass checks that and
//      finds where each window starts.  Otherwise the edges become u64
//      elements, partitioned by the window's bits alone (stable 8-bit
//      passes: two for 2^16 windows).
//   2. Lists.  One wave orders a window of up to 1024 edges by b, in
//      registers, and reads its list off the sorted keys.  A longer window
//      takes a workgroup, which sets its masks' bits in an LDS byte per b
//      (128K of them at a time) and reads them off in order, with no sort
//      however long the window is.  For BCSC each list is then reordered by
//      degree, the mask's population.  Where one window would keep its
//      workgroup longer than a sort of all edges takes, they are sorted and
//      the lists read off an edge a thread.
//   3. The lists' lengths give the block offsets (one scan), and one pass
//      over the edges' positions writes blocks, bitmaps and value offsets.
// The host waits once (and once more where the order check decides the route),
// to learn the block count; outputs are sized before by what E edges can need
// (the largest after one more wait).
//
// Bound by launches and by each pass's chain of loads at 1M edges, by the
// lists' instructions at 100M.  The sort of whole 36-bit keys with an edge
// permutation (BCSR) and the SWTCF conversion with one window a super-window
// (BCSC) that this replaced made 50 launches each and wrote 40 bytes an edge
// between their passes.  One build, host time with its allocations, R-MAT
// graphs in row order:
//   169k nodes, 1.17M edges: BCSR 0.45 -> 0.11 ms, BCSC 1.2 -> 0.15 ms
//   233k nodes, 114M edges:  BCSR 12.7 -> 4.4 ms, BCSC 36 -> 6.5 ms
// (shuffled, BCSR 0.44 -> 0.23 ms and 13.0 -> 6.1 ms).
#include <algorithm>
#include <cstring>
#include <type_traits>

#include "../../include/tcc_spmm_cnic.h"
#include "../../include/tcc_swtcf.h"
#include "common.hpp"
#include "primitives.hpp"
#include "scratch.hpp"

namespace tcc {
namespace {

constexpr unsigned kThreads = 256;

inline unsigned ceil_log2(std::uint64_t x) {
    unsigned b = 0;
    while ((1ull << b) < x) ++b;
    return b;
}

inline std::size_t align_up(std::size_t x) { return (x + 255) & ~std::size_t(255); }

// ---------------------------------------------------------------- edges

// The COO as (a, b): windows of 8 consecutive a, lists of b.  With phases > 1
// (BCSR) the window of an edge is phase(b) * windowsPerPhase + a / 8, where
// column b is in phase b * phases / numB: the matrix is built as its column
// slices stacked vertically.
struct Coo {
    const std::uint32_t* a;
    const std::uint32_t* b;
    std::uint32_t E, numA, numB;
    std::uint32_t phases, windowsPerPhase;
    unsigned bBits;
};

struct Edge {
    std::uint32_t w, b, lo;  // window, list index, a % 8
};

// Flag words (device): what went wrong or was found.
constexpr unsigned kFlagRange = 0, kFlagUngrouped = 1, kFlagDuplicate = 2, kNumMid = 3, kNumBig = 4, kFlagTooLong = 5;

// Edge i; indices out of range become (0, 0) and set `bad`.
__device__ __forceinline__ Edge coo_edge(const Coo& c, std::uint32_t i, bool& bad) {
    std::uint32_t a = c.a[i], b = c.b[i];
    if (a >= c.numA || b >= c.numB) {
        bad = true;
        a = 0;
        b = 0;
    }
    std::uint32_t w = a >> 3;
    if (c.phases > 1)
        w += static_cast<std::uint32_t>(static_cast<std::uint64_t>(b) * c.phases / c.numB) * c.windowsPerPhase;
    return Edge{w, b, a & 7u};
}

__device__ __forceinline__ std::uint64_t pack_edge(const Edge& e, unsigned bBits) {
    return (((static_cast<std::uint64_t>(e.w) << bBits) | e.b) << 3) | e.lo;
}

__device__ __forceinline__ Edge unpack_edge(std::uint64_t k, unsigned bBits) {
    const std::uint32_t mask = bBits >= 32 ? 0xFFFFFFFFu : (1u << bBits) - 1u;
    return Edge{static_cast<std::uint32_t>(k >> (bBits + 3)), static_cast<std::uint32_t>(k >> 3) & mask,
                static_cast<std::uint32_t>(k) & 7u};
}

// Edge i of the grouped order: the partitioned elements, or the COO itself.
template <bool KEYS>
__device__ __forceinline__ Edge grouped_edge(const Coo& c, const std::uint64_t* keys, std::uint32_t i) {
    if constexpr (KEYS) {
        return unpack_edge(keys[i], c.bBits);
    } else {
        bool bad = false;
        return coo_edge(c, i, bad);
    }
}

template <bool KEYS>
__device__ __forceinline__ std::uint32_t grouped_window(const Coo& c, const std::uint64_t* keys, std::uint32_t i) {
    if constexpr (KEYS) return static_cast<std::uint32_t>(keys[i] >> (c.bBits + 3));
    else return c.a[i] >> 3;  // in range, and one phase: checked before
}

// Window starts: the thread of edge i writes i to every window after its
// predecessor's up to its own (thread E: to all that are left), so
// winStart[w] is the first edge of window w or of the next one with edges.
// Runs of empty windows are filled by the whole wave.  Without KEYS this is
// also the check of the COO: indices in range, windows never decreasing (if
// they do, winStart is not used).
template <bool KEYS>
__global__ void __launch_bounds__(kThreads) window_starts_kernel(Coo c, const std::uint64_t* __restrict__ keys,
                                                                std::uint32_t RW, std::uint32_t* __restrict__ winStart,
                                                                std::uint32_t* __restrict__ flags) {
    const std::uint64_t i = static_cast<std::uint64_t>(blockIdx.x) * kThreads + threadIdx.x;
    bool bad = false;
    std::int64_t w = -1, before = -1;  // this edge's window, the previous edge's
    if (i < c.E) {
        if constexpr (KEYS) w = grouped_window<true>(c, keys, static_cast<std::uint32_t>(i));
        else w = coo_edge(c, static_cast<std::uint32_t>(i), bad).w;
    } else if (i == c.E) {
        w = RW;
    }
    if (i > 0 && i <= c.E) {
        bool ignore = false;
        if constexpr (KEYS) before = grouped_window<true>(c, keys, static_cast<std::uint32_t>(i - 1));
        else before = coo_edge(c, static_cast<std::uint32_t>(i - 1), ignore).w;
    }
    if constexpr (!KEYS) {
        raise_flag(&flags[kFlagRange], bad);
        raise_flag(&flags[kFlagUngrouped], i < c.E && w < before);
    }
    std::int64_t gap = i <= c.E ? w - before : 0;
    if constexpr (!KEYS) {
        // no starts from a COO seen to be ungrouped: its steps up would fill
        // nearly every window again and again
        if (__ballot(i < c.E && w < before) != 0 ||
            __hip_atomic_load(&flags[kFlagUngrouped], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u)
            gap = 0;
    }
    if (gap == 1) winStart[w] = static_cast<std::uint32_t>(i);
    std::uint64_t todo = __ballot(gap > 1);
    while (todo) {
        const int l = __builtin_ctzll(todo);
        todo &= todo - 1;
        const std::uint32_t first = static_cast<std::uint32_t>(__shfl(static_cast<int>(before), l)) + 1;
        const std::uint32_t last = static_cast<std::uint32_t>(__shfl(static_cast<int>(w), l));
        const std::uint32_t at = static_cast<std::uint32_t>(__shfl(static_cast<int>(i), l));
        for (std::uint64_t x = static_cast<std::uint64_t>(first) + __lane_id(); x <= last; x += kWave)
            winStart[x] = at;
    }
}

// ---------------------------------------------------------------- partition

// Elements of the first pass, from the COO (ranges checked), for the
// partition by the window's digits.
struct CooLoad {
    Coo c;
    std::uint32_t* flags;
    __device__ __forceinline__ void load(std::uint64_t first, std::uint64_t (&k)[kPrimRounds], bool& bad) const {
        std::uint32_t a[kPrimRounds], b[kPrimRounds];
        const std::uint64_t last = c.E - 1;
#pragma unroll
        for (int r = 0; r < kPrimRounds; ++r) {
            const std::uint64_t i = first + r * kWave < last ? first + r * kWave : last;
            a[r] = c.a[i];
            b[r] = c.b[i];
        }
#pragma unroll
        for (int r = 0; r < kPrimRounds; ++r) {
            if (a[r] >= c.numA || b[r] >= c.numB) {
                bad = true;
                a[r] = 0;
                b[r] = 0;
            }
            std::uint32_t w = a[r] >> 3;
            if (c.phases > 1)
                w += static_cast<std::uint32_t>(static_cast<std::uint64_t>(b[r]) * c.phases / c.numB) *
                     c.windowsPerPhase;
            k[r] = pack_edge(Edge{w, b[r], a[r] & 7u}, c.bBits);
        }
    }
    __device__ __forceinline__ void report(bool bad) const { raise_flag(&flags[kFlagRange], bad); }
};

// ---------------------------------------------------------------- lists

// Every window's list, at the positions of its edges (winStart[w] on, a list
// being at most as long as its window): the final order's b, mask and the
// number of the window's entries before (value offsets); for BCSC also b in
// ascending order (sB, with its mask while a long window is reordered) and
// each one's place in the final order, which the values are placed by.
struct Lists {
    const std::uint32_t* winStart;  // [RW + 1]
    std::uint32_t RW;
    std::uint32_t* length;  // [RW], zeroed before
    std::uint32_t* b;       // [E]
    std::uint8_t* mask;     // [E]
    std::uint32_t* before;  // [E]
    std::uint32_t* sB;      // [E] (BCSC)
    std::uint8_t* sMask;    // [E] (BCSC)
    std::uint32_t* sPlace;  // [E] (BCSC with values, else null)
    std::uint32_t* mid;     // windows of at most kMid edges for the second pass, flags[kNumMid] of them
    std::uint32_t* big;     // longer ones, flags[kNumBig] of them
    std::uint32_t longest;  // edges of a window that one workgroup may take
    std::uint32_t* flags;
};

// Windows of at most kShort edges are ordered by one wave of the first pass.
// Of the others, those of at most kMid take one wave, longer ones a
// workgroup, in the second.
constexpr unsigned kShort = 256;
constexpr unsigned kMid = 1024;
constexpr unsigned kListWaves = 8;

// Value of the lane whose number differs in bit D.
template <int D>
__device__ __forceinline__ std::uint32_t xor_lane(std::uint32_t v) {
    if constexpr (D == 32) return static_cast<std::uint32_t>(__shfl_xor(static_cast<int>(v), 32, kWave));
    else return static_cast<std::uint32_t>(__builtin_amdgcn_ds_swizzle(static_cast<int>(v), 0x1F | (D << 10)));
}

template <int D>
__device__ __forceinline__ std::uint64_t xor_lane(std::uint64_t v) {
    return (static_cast<std::uint64_t>(xor_lane<D>(static_cast<std::uint32_t>(v >> 32))) << 32) |
           xor_lane<D>(static_cast<std::uint32_t>(v));
}

// One wave sorts 64 V keys ascending in registers: element V * lane + r is
// k[r], so a bitonic step of stride below V exchanges registers and a longer
// one lanes.  (S, J): the step of stride 2^J in the merge of 2^S elements.
// About 4 instructions an element and step: 21 steps at 64 keys, 66 at 2048,
// against 4-5 passes of about 60 instructions for a radix sort in LDS.
template <int S, int J, typename K, int V>
__device__ __forceinline__ void sort_steps(K (&k)[V]) {
    constexpr int kLogV = V == 1 ? 0 : V == 2 ? 1 : V == 4 ? 2 : V == 8 ? 3 : 4;
    constexpr int kLogN = kLogV + 6;
    const unsigned lane = __lane_id();
    if constexpr (J < kLogV) {
#pragma unroll
        for (int r = 0; r < V; ++r) {
            constexpr int kStride = 1 << J;
            if (r & kStride) continue;
            const bool up = S < kLogV ? ((r >> S) & 1) == 0 : ((lane >> (S < kLogV ? 0 : S - kLogV)) & 1u) == 0;
            const K x = k[r], y = k[r | kStride];
            const K lo = x < y ? x : y, hi = x < y ? y : x;
            k[r] = up ? lo : hi;
            k[r | kStride] = up ? hi : lo;
        }
    } else {
        constexpr int D = 1 << (J - kLogV);
        const bool keepMin = ((lane & D) == 0) == (((lane >> (S - kLogV)) & 1u) == 0);
#pragma unroll
        for (int r = 0; r < V; ++r) {
            const K other = xor_lane<D>(k[r]);
            const K lo = k[r] < other ? k[r] : other, hi = k[r] < other ? other : k[r];
            k[r] = keepMin ? lo : hi;
        }
    }
    if constexpr (J > 0) sort_steps<S, J - 1, K, V>(k);
    else if constexpr (S < kLogN) sort_steps<S + 1, S, K, V>(k);
}

// The staged keys of a window, one word of padding every 32 (a lane's V
// consecutive keys would otherwise share their banks).
__host__ __device__ constexpr unsigned staged(unsigned i) { return i + (i >> 5); }

// Loads, sorts and stages window [begin, begin + n), n <= 64 V.
template <bool KEYS, typename K, int V>
__device__ __forceinline__ void sort_window(const Coo& c, const std::uint64_t* __restrict__ keys, std::uint32_t begin,
                                            unsigned n, K* __restrict__ stage) {
    const unsigned lane = __lane_id();
    K k[V];
#pragma unroll
    for (int r = 0; r < V; ++r) {
        const unsigned i = r * kWave + lane;
        const Edge e = grouped_edge<KEYS>(c, keys, begin + min(i, n - 1));
        k[r] = i < n ? (static_cast<K>(e.b) << 3) | e.lo : ~static_cast<K>(0);
    }
    sort_steps<1, 0, K, V>(k);
#pragma unroll
    for (int r = 0; r < V; ++r)
        if (V * lane + r < n) stage[staged(V * lane + r)] = k[r];
    __builtin_amdgcn_wave_barrier();
}

// The list of a staged, sorted window: its entries are the runs of equal b
// (at most 8 edges, one per a % 8).
template <typename K, bool DEGREE>
__device__ __forceinline__ void write_list(const Lists& L, std::uint32_t w, std::uint32_t begin, unsigned n,
                                           K* __restrict__ stage, std::uint8_t* __restrict__ masks) {
    const unsigned lane = __lane_id();
    const std::uint64_t lt = lanemask_lt();
    std::uint32_t run = 0;
    bool dup = false;
    K last = 0;  // the key before the round's first
    for (unsigned i0 = 0; i0 < n; i0 += kWave) {
        const unsigned i = i0 + lane;
        const K key = i < n ? stage[staged(i)] : ~static_cast<K>(0);
        const K prev = lane == 0 ? last : (i < n ? stage[staged(i - 1)] : static_cast<K>(0));
        const bool entry = i < n && (i == 0 || (prev >> 3) != (key >> 3));
        dup |= i < n && i > 0 && prev == key;
        std::uint32_t mask = 1u << static_cast<unsigned>(key & 7u);
        if (entry) {
            for (unsigned q = 1; q < 8; ++q) {
                if (i + q >= n) break;
                const K x = stage[staged(i + q)];
                if ((x >> 3) != (key >> 3)) break;
                mask |= 1u << static_cast<unsigned>(x & 7u);
            }
        }
        if constexpr (sizeof(K) == 4)
            last = static_cast<K>(__builtin_amdgcn_readlane(static_cast<int>(key), kWave - 1));
        else
            last = __shfl(key, kWave - 1, kWave);
        __builtin_amdgcn_wave_barrier();  // every read of the round is before the writes below
        const std::uint64_t eb = __ballot(entry);
        const std::uint32_t rank = run + static_cast<std::uint32_t>(__popcll(eb & lt));
        run += static_cast<std::uint32_t>(__popcll(eb));
        if (entry) {
            const std::uint32_t b = static_cast<std::uint32_t>(key >> 3);
            if constexpr (DEGREE) {
                // compacted in place: rank <= i
                stage[staged(rank)] = key;
                masks[rank] = static_cast<std::uint8_t>(mask);
                if (L.sPlace) L.sB[begin + rank] = b;
            } else {
                L.b[begin + rank] = b;
                L.mask[begin + rank] = static_cast<std::uint8_t>(mask);
                L.before[begin + rank] = i;
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
    raise_flag(&L.flags[kFlagDuplicate], dup);
    if (lane == 0) L.length[w] = run;
    if constexpr (DEGREE) {
        // stable by degree, 8 first: counts, the degrees' places, ranks
        std::uint32_t place[8], before[8];
#pragma unroll
        for (unsigned k = 0; k < 8; ++k) place[k] = 0;
        for (unsigned i0 = 0; i0 < run; i0 += kWave) {
            const unsigned d = i0 + lane < run ? 8u - static_cast<unsigned>(__popc(masks[i0 + lane])) : 8u;
#pragma unroll
            for (unsigned k = 0; k < 8; ++k) place[k] += static_cast<std::uint32_t>(__popcll(__ballot(d == k)));
        }
        std::uint32_t p = 0, q = 0;
#pragma unroll
        for (unsigned k = 0; k < 8; ++k) {
            const std::uint32_t m = place[k];
            place[k] = p;
            before[k] = q - (8u - k) * p;  // edges before place x of the degree: before + (8 - k) x
            p += m;
            q += (8u - k) * m;
        }
        for (unsigned i0 = 0; i0 < run; i0 += kWave) {
            const unsigned i = i0 + lane;
            const unsigned m = i < run ? masks[i] : 0u;
            const unsigned d = 8u - static_cast<unsigned>(__popc(m));
            std::uint32_t at = 0, ed = 0;
#pragma unroll
            for (unsigned k = 0; k < 8; ++k) {
                const std::uint64_t same = __ballot(d == k);
                if (d == k) {
                    at = place[k] + static_cast<std::uint32_t>(__popcll(same & lt));
                    ed = before[k] + (8u - k) * at;
                }
                place[k] += static_cast<std::uint32_t>(__popcll(same));
            }
            if (i < run) {
                L.b[begin + at] = static_cast<std::uint32_t>(stage[staged(i)] >> 3);
                L.mask[begin + at] = static_cast<std::uint8_t>(m);
                L.before[begin + at] = ed;
                if (L.sPlace) L.sPlace[begin + i] = at;
            }
        }
    }
}

// One wave per window; windows too long for it go to their pass's list.
template <bool KEYS, bool DEGREE, typename K>
__global__ void __launch_bounds__(kListWaves * kWave) short_lists_kernel(Coo c, const std::uint64_t* __restrict__ keys,
                                                                        Lists L) {
    __shared__ K stage[kListWaves][staged(kShort)];
    __shared__ std::uint8_t masks[kListWaves][kShort];
    __shared__ std::uint32_t listAt[2];  // the workgroup's places in the two lists
    __shared__ std::uint8_t kind[kListWaves];
    const unsigned wave = threadIdx.x / kWave;
    const std::uint64_t w64 = static_cast<std::uint64_t>(blockIdx.x) * kListWaves + wave;
    const std::uint32_t w = static_cast<std::uint32_t>(min<std::uint64_t>(w64, L.RW - 1));
    const std::uint32_t begin = uniform(L.winStart[w]);
    const std::uint32_t n = w64 < L.RW ? uniform(L.winStart[w + 1]) - begin : 0u;
    // one atomic per workgroup and list: those on one address queue up
    // (4,096 of them took 50 us)
    if (__lane_id() == 0) kind[wave] = n <= kShort ? 0 : n <= kMid ? 1 : 2;
    __syncthreads();
    if (threadIdx.x < 2) {
        std::uint32_t k = 0;
        for (unsigned v = 0; v < kListWaves; ++v) k += kind[v] == threadIdx.x + 1;
        if (k) listAt[threadIdx.x] = atomicAdd(&L.flags[threadIdx.x ? kNumBig : kNumMid], k);
    }
    __syncthreads();
    if (n > kShort) {
        std::uint32_t before = 0;
        for (unsigned v = 0; v < wave; ++v) before += kind[v] == kind[wave];
        if (__lane_id() == 0) {
            if (n <= kMid) {
                L.mid[listAt[0] + before] = w;
            } else {
                L.big[listAt[1] + before] = w;
                if (n > L.longest) L.flags[kFlagTooLong] = 1;
            }
        }
        return;
    }
    if (n == 0) return;
    if (n <= 64) sort_window<KEYS, K, 1>(c, keys, begin, n, stage[wave]);
    else if (n <= 128) sort_window<KEYS, K, 2>(c, keys, begin, n, stage[wave]);
    else sort_window<KEYS, K, 4>(c, keys, begin, n, stage[wave]);
    write_list<K, DEGREE>(L, w, begin, n, stage[wave], masks[wave]);
}

// Exclusive scan over the workgroup of one value per thread; waveSum holds
// one word per wave and is free again after the call.
template <unsigned WAVES>
__device__ __forceinline__ std::uint32_t block_scan(std::uint32_t v, std::uint32_t* waveSum, std::uint32_t& all) {
    const unsigned lane = __lane_id(), wave = threadIdx.x / kWave;
    const std::uint32_t inc = wave_inclusive_scan(v);
    if (lane == kWave - 1) waveSum[wave] = inc;
    __syncthreads();
    std::uint32_t off = inc - v;
    all = 0;
#pragma unroll
    for (unsigned w = 0; w < WAVES; ++w) {
        if (w < wave) off += waveSum[w];
        all += waveSum[w];
    }
    __syncthreads();
    return off;
}

// The other windows: 1024-thread workgroups that first take the long ones,
// one each at a time from the first workgroup on, and then the mid ones, one
// wave each from the last workgroup back, so that few wait for a long one.
//
// Long: an LDS byte per b of a slice of 128K holds its mask and a bit its
// use, both set with LDS atomics whatever the order of the window's edges;
// wave v then reads off the 8K columns of its part in order, 32 a lane by
// the set bits (and clears them).
constexpr unsigned kSlice = 131072;
constexpr unsigned kLongThreads = 1024;
constexpr unsigned kLongWaves = kLongThreads / kWave;
constexpr unsigned kUseWords = kSlice / 32;
constexpr unsigned kLongSteps = kUseWords / kLongThreads;  // 64 words a wave and step

// A workgroup goes through a long window once for each slice (0.13 to 0.7 ns an
// edge and slice) and no other can help it.  Where that is more for the longest
// window than sorting the whole COO takes (0.1 ms and 0.06 ns an edge; BCSC
// about twice that), the lists are made of the sorted COO instead.  Builds in
// ms, a workgroup a window : all sorted: 8 x 1M with 2M edges BCSR 12.0 : 0.19,
// 64 x 4M with 8M edges 21.4 : 0.53; 2M x 64 with 8M edges BCSC 4.7 : 0.71; a
// 1M-node graph of 8M edges with one row and one column joined to all BCSR
// 8.1 : 0.90, BCSC 5.0 : 1.48 (0.45 and 0.64 without them).
inline std::uint32_t longest_window(std::uint64_t E, std::uint32_t numB) {
    return static_cast<std::uint32_t>(((1ull << 18) + E / 4) / ((numB - 1) / kSlice + 1));
}

template <typename K>
constexpr unsigned other_lists_lds() {
    const unsigned mid = kLongWaves * (staged(kMid) * sizeof(K) + kMid), big = kSlice + 4 * kUseWords;
    return mid > big ? mid : big;
}

template <bool KEYS, bool DEGREE, typename K>
__global__ void __launch_bounds__(kLongThreads) other_lists_kernel(Coo c, const std::uint64_t* __restrict__ keys,
                                                                  Lists L) {
    extern __shared__ __attribute__((aligned(16))) std::uint32_t lds[];
    __shared__ std::uint32_t waveSum[kLongWaves], waveSum2[kLongWaves];
    __shared__ std::uint32_t degCount[kLongWaves][8];
    __shared__ std::uint32_t used[1u << 10];  // slices with edges (2^15 of 2^17 cover any b)
    const unsigned lane = __lane_id(), wave = threadIdx.x / kWave;
    const std::uint64_t lt = lanemask_lt();
    const std::uint32_t numBig = L.flags[kNumBig], numMid = L.flags[kNumMid];
    if (L.flags[kFlagTooLong]) return;
    std::uint32_t* const bytes = lds;              // [kSlice / 4] masks
    std::uint32_t* const use = lds + kSlice / 4;   // [kUseWords]
    if (blockIdx.x < numBig) {
        for (unsigned i = threadIdx.x; i < (kSlice + 4 * kUseWords) / 16; i += kLongThreads)
            reinterpret_cast<vu4*>(lds)[i] = vu4{0, 0, 0, 0};
    }
    for (std::uint32_t g = blockIdx.x; g < numBig; g += gridDim.x) {
        const std::uint32_t w = L.big[g];
        const std::uint32_t begin = L.winStart[w], n = L.winStart[w + 1] - begin;
        std::uint32_t entries = 0, edges = 0;  // of the slices so far
        bool dup = false;
        const bool choose = c.numB > 4 * kSlice;  // fewer are swept without a look
        if (choose) {
            used[threadIdx.x] = 0;
            __syncthreads();
            for (std::uint32_t i = threadIdx.x; i < n; i += kLongThreads) {
                const std::uint32_t sl = grouped_edge<KEYS>(c, keys, begin + i).b / kSlice;
                atomicOr(&used[sl >> 5], 1u << (sl & 31u));
            }
        }
        __syncthreads();
        for (std::uint64_t s0 = 0; s0 < c.numB; s0 += kSlice) {
            const std::uint32_t sl = static_cast<std::uint32_t>(s0 / kSlice);
            if (choose && ((used[sl >> 5] >> (sl & 31u)) & 1u) == 0) continue;
            for (std::uint32_t i0 = threadIdx.x; i0 < n; i0 += 4 * kLongThreads) {
                Edge e[4];
#pragma unroll
                for (unsigned q = 0; q < 4; ++q)
                    e[q] = grouped_edge<KEYS>(c, keys, begin + min(i0 + q * kLongThreads, n - 1));
#pragma unroll
                for (unsigned q = 0; q < 4; ++q) {
                    const std::uint64_t x = e[q].b - s0;  // wraps below the slice: then >= kSlice
                    if (i0 + q * kLongThreads < n && x < kSlice) {
                        const std::uint32_t bit = 1u << (8 * (x & 3u) + e[q].lo);
                        dup |= (atomicOr(&bytes[x >> 2], bit) & bit) != 0;
                        atomicOr(&use[x >> 5], 1u << (x & 31u));
                    }
                }
            }
            __syncthreads();
            const std::uint8_t* mask8 = reinterpret_cast<const std::uint8_t*>(bytes);
            std::uint32_t bits[kLongSteps], both[kLongSteps];  // both: entries | edges << 16 of the lane's word
            std::uint32_t myEntries = 0, myEdges = 0;
#pragma unroll
            for (unsigned st = 0; st < kLongSteps; ++st) {
                const unsigned word = (wave * kLongSteps + st) * kWave + lane;
                bits[st] = use[word];
                std::uint32_t ed = 0;
                for (std::uint32_t m = bits[st]; m; m &= m - 1) ed += __popc(mask8[32 * word + __builtin_ctz(m)]);
                both[st] = static_cast<std::uint32_t>(__popc(bits[st])) | (ed << 16);
                myEntries += both[st] & 0xFFFFu;
                myEdges += ed;
            }
            const std::uint32_t allEntries = wave_inclusive_scan(myEntries), allEdges = wave_inclusive_scan(myEdges);
            if (lane == kWave - 1) {
                waveSum[wave] = allEntries;
                waveSum2[wave] = allEdges;
            }
            __syncthreads();
            std::uint32_t at = begin + entries, ed = edges;
#pragma unroll
            for (unsigned v = 0; v < kLongWaves; ++v) {
                if (v < wave) {
                    at += waveSum[v];
                    ed += waveSum2[v];
                }
                entries += waveSum[v];
                edges += waveSum2[v];
            }
#pragma unroll
            for (unsigned st = 0; st < kLongSteps; ++st) {
                const unsigned word = (wave * kLongSteps + st) * kWave + lane;
                const std::uint32_t inc = wave_inclusive_scan(both[st]);  // at most 2048 and 16384
                std::uint32_t p = at + ((inc - both[st]) & 0xFFFFu), q = ed + ((inc - both[st]) >> 16);
                for (std::uint32_t m = bits[st]; m; m &= m - 1) {
                    const unsigned x = 32 * word + __builtin_ctz(m);
                    const std::uint32_t b = static_cast<std::uint32_t>(s0) + x, mask = mask8[x];
                    if constexpr (DEGREE) {
                        L.sB[p] = b;
                        L.sMask[p] = static_cast<std::uint8_t>(mask);
                    } else {
                        L.b[p] = b;
                        L.mask[p] = static_cast<std::uint8_t>(mask);
                        L.before[p] = q;
                    }
                    ++p;
                    q += __popc(mask);
                }
                if (bits[st]) {
                    use[word] = 0;
                    reinterpret_cast<vu4*>(bytes)[2 * word] = vu4{0, 0, 0, 0};
                    reinterpret_cast<vu4*>(bytes)[2 * word + 1] = vu4{0, 0, 0, 0};
                }
                const std::uint32_t tot = static_cast<std::uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(inc), kWave - 1));
                at += tot & 0xFFFFu;
                ed += tot >> 16;
            }
            __syncthreads();
        }
        raise_flag(&L.flags[kFlagDuplicate], dup);
        if (threadIdx.x == 0) L.length[w] = entries;
        if constexpr (DEGREE) {
            // stable by degree, 8 first.  Wave v takes the entries of its
            // sixteenth of the list: counts per degree, then ranks.
            const std::uint32_t span = ((entries + kLongWaves - 1) / kLongWaves + kWave - 1) / kWave * kWave;
            const std::uint32_t e0 = min(wave * span, entries), e1 = min(e0 + span, entries);
            std::uint32_t count[8] = {0, 0, 0, 0, 0, 0, 0, 0};
            for (std::uint32_t i = e0; i < e1; i += kWave) {
                const unsigned m = i + lane < e1 ? L.sMask[begin + i + lane] : 0u;
                const unsigned d = 8u - static_cast<unsigned>(__popc(m));  // 8 for none
#pragma unroll
                for (unsigned k = 0; k < 8; ++k) count[k] += static_cast<std::uint32_t>(__popcll(__ballot(d == k)));
            }
            if (lane < 8) {
                std::uint32_t mine = 0;
#pragma unroll
                for (unsigned k = 0; k < 8; ++k) mine = lane == k ? count[k] : mine;
                degCount[wave][lane] = mine;
            }
            __syncthreads();
            std::uint32_t place[8], before[8];  // of degree 8 - k: this wave's next place, the edges before place 0
            std::uint32_t p = 0, q = 0;
#pragma unroll
            for (unsigned k = 0; k < 8; ++k) {
                std::uint32_t own = 0, all = 0;
#pragma unroll 1
                for (unsigned v = 0; v < kLongWaves; ++v) {
                    const std::uint32_t x = degCount[v][k];
                    if (v < wave) own += x;
                    all += x;
                }
                place[k] = p + own;
                before[k] = q - (8u - k) * p;  // edges before place x of the degree: before + (8 - k) x
                p += all;
                q += (8u - k) * all;
            }
            for (std::uint32_t i = e0; i < e1; i += kWave) {
                const bool valid = i + lane < e1;
                const unsigned m = valid ? L.sMask[begin + i + lane] : 0u;
                const std::uint32_t b = valid ? L.sB[begin + i + lane] : 0u;
                const unsigned d = 8u - static_cast<unsigned>(__popc(m));
                std::uint32_t at = 0, ed = 0;
#pragma unroll
                for (unsigned k = 0; k < 8; ++k) {
                    const std::uint64_t same = __ballot(d == k);
                    if (d == k) {
                        at = place[k] + static_cast<std::uint32_t>(__popcll(same & lt));
                        ed = before[k] + (8u - k) * at;
                    }
                    place[k] += static_cast<std::uint32_t>(__popcll(same));
                }
                if (valid) {
                    L.b[begin + at] = b;
                    L.mask[begin + at] = static_cast<std::uint8_t>(m);
                    L.before[begin + at] = ed;
                    if (L.sPlace) L.sPlace[begin + i + lane] = at;
                }
            }
        }
        __syncthreads();  // the shared arrays are free for the next window
    }
    // mid windows
    K* const stage = reinterpret_cast<K*>(lds) + wave * staged(kMid);
    std::uint8_t* const masks =
        reinterpret_cast<std::uint8_t*>(reinterpret_cast<K*>(lds) + kLongWaves * staged(kMid)) + wave * kMid;
    for (std::uint32_t g = (gridDim.x - 1 - blockIdx.x) * kLongWaves + wave; g < numMid; g += gridDim.x * kLongWaves) {
        const std::uint32_t w = uniform(L.mid[g]);
        const std::uint32_t begin = uniform(L.winStart[w]), n = uniform(L.winStart[w + 1]) - begin;
        if (n <= 512) sort_window<KEYS, K, 8>(c, keys, begin, n, stage);
        else sort_window<KEYS, K, 16>(c, keys, begin, n, stage);
        write_list<K, DEGREE>(L, w, begin, n, stage, masks);
    }
}

// ---------------------------------------------------------------- lists of a sorted COO

// 1 where a list entry starts: the first edge of its (window, b).
__global__ void __launch_bounds__(kThreads) entry_heads_kernel(const std::uint64_t* __restrict__ keys, std::uint32_t E,
                                                              std::uint32_t* __restrict__ heads) {
    const std::uint64_t i = static_cast<std::uint64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (i < E) heads[i] = i == 0 || (keys[i] >> 3) != (keys[i - 1] >> 3);
}

// The lists of the edges in (window, b, a % 8) order, an edge a thread (for
// BCSC in that order still); pos: the entries that start before each edge.
template <bool DEGREE>
__global__ void __launch_bounds__(kThreads) sorted_lists_kernel(const std::uint64_t* __restrict__ keys,
                                                               const std::uint32_t* __restrict__ pos, std::uint32_t E,
                                                               unsigned bBits, Lists L) {
    const std::uint64_t i = static_cast<std::uint64_t>(blockIdx.x) * kThreads + threadIdx.x;
    bool dup = false;
    if (i < E) {
        const std::uint64_t k = keys[i], prev = i > 0 ? keys[i - 1] : ~k;
        const Edge e = unpack_edge(k, bBits);
        const std::uint32_t begin = L.winStart[e.w], first = pos[begin];
        const bool head = (k >> 3) != (prev >> 3);
        dup = k == prev;
        if (head) {
            std::uint32_t mask = 1u << e.lo;
            for (unsigned q = 1; q < 8 && i + q < E; ++q) {
                const std::uint64_t x = keys[i + q];
                if ((x >> 3) != (k >> 3)) break;
                mask |= 1u << static_cast<unsigned>(x & 7u);
            }
            const std::uint32_t at = begin + (pos[i] - first);
            if constexpr (DEGREE) {
                L.sB[at] = e.b;
                L.sMask[at] = static_cast<std::uint8_t>(mask);
            } else {
                L.b[at] = e.b;
                L.mask[at] = static_cast<std::uint8_t>(mask);
                L.before[at] = static_cast<std::uint32_t>(i) - begin;
            }
        }
        if (i + 1 == L.winStart[e.w + 1]) L.length[e.w] = pos[i] + (head ? 1u : 0u) - first;
    }
    raise_flag(&L.flags[kFlagDuplicate], dup);
}

// BCSC: list position i's element for the order by degree, (window, 8 - degree,
// i); the positions past a list's end stay behind its entries as degree 1.
__global__ void __launch_bounds__(kThreads) degree_elems_kernel(const std::uint64_t* __restrict__ keys, std::uint32_t E,
                                                               unsigned bBits, Lists L,
                                                               std::uint64_t* __restrict__ elems) {
    const std::uint64_t i = static_cast<std::uint64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (i >= E) return;
    const std::uint32_t w = unpack_edge(keys[i], bBits).w;
    const bool entry = static_cast<std::uint32_t>(i) - L.winStart[w] < L.length[w];
    const unsigned d = entry ? 8u - static_cast<unsigned>(__popc(L.sMask[i])) : 7u;
    elems[i] = (((static_cast<std::uint64_t>(w) << 3) | d) << 32) | i;
}

// The entry at each place of that order: its degree (0 past a list's end), and
// after their scan, which counts a window's edges up to its end, the list.
struct ByDegree {
    std::uint32_t w, i, degree;
};

__device__ __forceinline__ ByDegree by_degree(std::uint64_t elem, const Lists& L) {
    ByDegree r;
    r.w = static_cast<std::uint32_t>(elem >> 35);
    r.i = static_cast<std::uint32_t>(elem);
    r.degree = r.i - L.winStart[r.w] < L.length[r.w] ? 8u - (static_cast<std::uint32_t>(elem >> 32) & 7u) : 0u;
    return r;
}

__global__ void __launch_bounds__(kThreads) degrees_kernel(const std::uint64_t* __restrict__ elems, std::uint32_t E,
                                                          Lists L, std::uint32_t* __restrict__ degree) {
    const std::uint64_t q = static_cast<std::uint64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (q < E) degree[q] = by_degree(elems[q], L).degree;
}

__global__ void __launch_bounds__(kThreads) degree_lists_kernel(const std::uint64_t* __restrict__ elems,
                                                               const std::uint32_t* __restrict__ edges, std::uint32_t E,
                                                               Lists L) {
    const std::uint64_t q = static_cast<std::uint64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (q >= E) return;
    const ByDegree r = by_degree(elems[q], L);
    if (r.degree == 0) return;
    const std::uint32_t begin = L.winStart[r.w];
    L.b[q] = L.sB[r.i];
    L.mask[q] = L.sMask[r.i];
    L.before[q] = edges[q] - begin;
    if (L.sPlace) L.sPlace[r.i] = static_cast<std::uint32_t>(q) - begin;
}

// ---------------------------------------------------------------- blocks

__global__ void blocks_per_window_kernel(const std::uint32_t* __restrict__ length, std::uint32_t n,
                                         std::uint32_t* __restrict__ blocks) {
    const std::uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) blocks[i] = (length[i] + 7) / 8;
}

// off[w] = blocks of the windows before w, off[RW] = all, in one workgroup
// (for window counts whose scan would be mostly launches).
constexpr std::uint32_t kOneScan = 65536;
__global__ void __launch_bounds__(1024) window_blocks_kernel(const std::uint32_t* __restrict__ length,
                                                            std::uint32_t RW, std::uint32_t* __restrict__ off) {
    __shared__ std::uint32_t waveSum[16];
    std::uint32_t run = 0;
    for (std::uint32_t base = 0; base < RW; base += 16384) {
        const std::uint32_t i0 = base + 16 * threadIdx.x;
        std::uint32_t v[16], s = 0, all;
#pragma unroll
        for (unsigned q = 0; q < 16; q += 4) {  // length is padded to 16 words past RW
            const vu4 x = load_global<vu4>(length + min(i0 + q, RW & ~3u));
            v[q] = x.x; v[q + 1] = x.y; v[q + 2] = x.z; v[q + 3] = x.w;
        }
#pragma unroll
        for (unsigned q = 0; q < 16; ++q) v[q] = i0 + q < RW ? (v[q] + 7) / 8 : 0u;
#pragma unroll
        for (unsigned q = 0; q < 16; ++q) s += v[q];
        std::uint32_t o = run + block_scan<16>(s, waveSum, all);
#pragma unroll
        for (unsigned q = 0; q < 16; q += 4) {  // off is 256-byte aligned
            vu4 x;
            x.x = o; o += v[q];
            x.y = o; o += v[q + 1];
            x.z = o; o += v[q + 2];
            x.w = o; o += v[q + 3];
            if (i0 + q + 4 <= RW) {
                *reinterpret_cast<vu4*>(off + i0 + q) = x;
            } else {
                if (i0 + q < RW) off[i0 + q] = x.x;
                if (i0 + q + 1 < RW) off[i0 + q + 1] = x.y;
                if (i0 + q + 2 < RW) off[i0 + q + 2] = x.z;
            }
        }
        run += all;
    }
    if (threadIdx.x == 0) off[RW] = run;
}

// 8 mask bits to the first bits of 8 bytes.
__device__ __forceinline__ std::uint64_t spread8(std::uint64_t x) {
    x = (x | (x << 28)) & 0x0000000F0000000Full;
    x = (x | (x << 14)) & 0x0003000300030003ull;
    return (x | (x << 7)) & 0x0101010101010101ull;
}

// The block count and the flags, for the host.
__device__ __forceinline__ void tell_host(const Lists& L, const std::uint32_t* off, std::uint32_t* mail) {
    mail[0] = off[L.RW];
    mail[1] = L.flags[kFlagRange];
    mail[2] = L.flags[kFlagDuplicate];
    mail[3] = L.flags[kFlagTooLong];
}

__global__ void tell_host_kernel(Lists L, const std::uint32_t* off, std::uint32_t* mail) { tell_host(L, off, mail); }

// Entry i (at its list's position) goes to its block; the first entry of a
// block also gathers the block's bitmap and pads it.  Thread 0 closes the
// value offsets and tells the host the block count and the flags.
template <bool KEYS, bool BCSC>
__global__ void __launch_bounds__(kThreads) emit_blocks_kernel(Coo c, const std::uint64_t* __restrict__ keys, Lists L,
                                                              const std::uint32_t* __restrict__ off,
                                                              std::uint32_t* __restrict__ tcOffset,
                                                              std::uint32_t* __restrict__ idx,
                                                              std::uint64_t* __restrict__ bits, std::uint32_t* mail) {
    const std::uint64_t i64 = static_cast<std::uint64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (i64 == 0) {
        tcOffset[off[L.RW]] = c.E;
        tell_host(L, off, mail);
    }
    if (i64 >= c.E) return;
    const std::uint32_t i = static_cast<std::uint32_t>(i64);
    const std::uint32_t w = grouped_window<KEYS>(c, keys, i);
    const std::uint32_t begin = L.winStart[w], len = L.length[w], j = i - begin;
    if (j >= len) return;
    const std::uint32_t blk = off[w] + j / 8;
    idx[static_cast<std::uint64_t>(blk) * 8 + (j & 7u)] = L.b[i];
    if (j & 7u) return;
    std::uint64_t bm = 0;
    for (unsigned q = 0; q < 8; ++q) {
        if (j + q < len) {
            const std::uint64_t m = L.mask[i + q];
            bm |= BCSC ? m << (8 * q) : spread8(m) << q;
        } else {
            idx[static_cast<std::uint64_t>(blk) * 8 + q] = TCC_SWTCF_INVALID_ROW_SLOT;
        }
    }
    bits[blk] = bm;
    tcOffset[blk] = begin + L.before[i];
}

// data[tcOffset[block] + rank of the entry's bit] = value of edge e, whose
// list entry is found by a search of its window's ascending b.
template <bool BCSC>
__global__ void __launch_bounds__(kThreads) place_values_kernel(Coo c, Lists L, const std::uint32_t* __restrict__ off,
                                                               const std::uint32_t* __restrict__ tcOffset,
                                                               const std::uint64_t* __restrict__ bits,
                                                               const float* __restrict__ val,
                                                               float* __restrict__ data) {
    const std::uint64_t e = static_cast<std::uint64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (e >= c.E) return;
    bool bad = false;
    const Edge x = coo_edge(c, static_cast<std::uint32_t>(e), bad);
    if (bad) return;
    const std::uint32_t begin = L.winStart[x.w], len = L.length[x.w];
    const std::uint32_t* list = (BCSC ? L.sB : L.b) + begin;
    std::uint32_t lo = 0, hi = len;
    while (lo < hi) {
        const std::uint32_t mid = (lo + hi) / 2;
        if (list[mid] < x.b) lo = mid + 1; else hi = mid;
    }
    if (lo >= len) return;  // duplicates or bad indices: the build is discarded
    const std::uint32_t j = BCSC ? L.sPlace[begin + lo] : lo;
    const std::uint32_t blk = off[x.w] + j / 8;
    const unsigned bit = BCSC ? (j & 7u) * 8 + x.lo : x.lo * 8 + (j & 7u);
    const std::uint32_t at = tcOffset[blk] + static_cast<std::uint32_t>(__popcll(bits[blk] & ((1ull << bit) - 1ull)));
    if (at < c.E) data[at] = val[e];
}

// ---------------------------------------------------------------- by conversion

// A BCSC of a COO with duplicate edges, or with the converter's errors to
// report: the SWTCF converter with one window per super-window (its row
// order is the BCSC's, a duplicate edge counting as another degree).
__global__ void popcount_kernel(const std::uint64_t* __restrict__ bits, std::uint32_t n,
                                std::uint32_t* __restrict__ out) {
    const std::uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = static_cast<std::uint32_t>(__popcll(bits[i]));
}

// BCSC from SWTCF(S=1): global destination of each tile row.
__global__ void bcsc_rows_kernel(const std::uint32_t* __restrict__ colWindowOffset, std::uint32_t CW,
                                 const std::uint32_t* __restrict__ swRowOffset,
                                 const std::uint32_t* __restrict__ swRows, const std::uint32_t* __restrict__ tileRowSlot,
                                 std::uint32_t T, std::uint32_t* __restrict__ sparseA2C,
                                 std::uint32_t* __restrict__ slotToLoc) {
    const std::uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= T * 8u) return;
    const std::uint32_t t = i / 8;
    std::uint32_t lo = 0, hi = CW;  // window of tile t: last w with colWindowOffset[w] <= t
    while (lo + 1 < hi) {
        const std::uint32_t mid = (lo + hi) / 2;
        if (colWindowOffset[mid] <= t) lo = mid; else hi = mid;
    }
    const std::uint32_t slot = tileRowSlot[i];
    if (slot == TCC_SWTCF_INVALID_ROW_SLOT) {
        sparseA2C[i] = TCC_SWTCF_INVALID_ROW_SLOT;
    } else {
        sparseA2C[i] = swRows[swRowOffset[lo] + slot];
        slotToLoc[swRowOffset[lo] + slot] = i;
    }
}

// Value placement for BCSC: edge (dst, src) -> tile row of dst in window src/8.
__global__ void bcsc_values_kernel(const std::uint32_t* __restrict__ dst, const std::uint32_t* __restrict__ src,
                                   const float* __restrict__ val, std::uint32_t E,
                                   const std::uint32_t* __restrict__ swRowOffset,
                                   const std::uint32_t* __restrict__ swRows,
                                   const std::uint32_t* __restrict__ slotToLoc,
                                   const std::uint64_t* __restrict__ bits, const std::uint32_t* __restrict__ tcOffset,
                                   float* __restrict__ data) {
    const std::uint32_t e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= E) return;
    const std::uint32_t w = src[e] >> 3, c = src[e] & 7u, d = dst[e];
    std::uint32_t lo = swRowOffset[w], hi = swRowOffset[w + 1];
    while (lo < hi) {
        const std::uint32_t mid = (lo + hi) / 2;
        if (swRows[mid] < d) lo = mid + 1; else hi = mid;
    }
    const std::uint32_t loc = slotToLoc[lo];
    const std::uint32_t t = loc / 8, bit = (loc & 7u) * 8 + c;
    data[tcOffset[t] + __popcll(bits[t] & ((1ull << bit) - 1ull))] = val ? val[e] : 1.0f;
}

}  // namespace
}  // namespace tcc

using namespace tcc;

namespace {

// The build's output arrays, in one allocation: off[RW + 1], tcOffset,
// idx, bits for at most maxB blocks, data[E] (with values).  A caller holds
// them for the matrix's life, and where windows share columns they have up to
// 8 times fewer blocks than their edges could fill: at most kMaxSlack of that
// is kept.  Arrays for kCountFirst bytes of blocks and more are allocated when
// the host knows their number (a wait more: 20 us, of 2 ms and more); smaller
// ones for what the edges could need, and moved to smaller ones at the end
// where that was much too much.
constexpr std::uint64_t kBlockBytes = 44, kMaxSlack = 32ull << 20, kCountFirst = 256ull << 20;
struct BlockArrays {
    char* base = nullptr;
    std::uint32_t *off = nullptr, *tcOffset = nullptr, *idx = nullptr;
    std::uint64_t* bits = nullptr;
    float* data = nullptr;

    hipError_t allocate(std::uint64_t RW, std::uint64_t maxB, std::uint64_t E, bool values) {
        const std::size_t sizes[5] = {align_up(4 * (RW + 1)), align_up(4 * (maxB + 1)), align_up(32 * std::max<std::uint64_t>(maxB, 1)),
                                      align_up(8 * std::max<std::uint64_t>(maxB, 1)),
                                      values ? align_up(4 * std::max<std::uint64_t>(E, 1)) : 0};
        const hipError_t e = pool_malloc(reinterpret_cast<void**>(&base),
                                               sizes[0] + sizes[1] + sizes[2] + sizes[3] + sizes[4]);
        if (e != hipSuccess) {
            base = nullptr;
            return e;
        }
        char* q = base;
        off = reinterpret_cast<std::uint32_t*>(q);
        tcOffset = reinterpret_cast<std::uint32_t*>(q += sizes[0]);
        idx = reinterpret_cast<std::uint32_t*>(q += sizes[1]);
        bits = reinterpret_cast<std::uint64_t*>(q += sizes[2]);
        data = values ? reinterpret_cast<float*>(q + sizes[3]) : nullptr;
        return hipSuccess;
    }
};

enum class Built { Ok, Range, Duplicate, TooLong };

// Builds the arrays of the COO over RW windows (E > 0).  A BCSR without
// phases checks whether the COO is grouped by window already; the source
// windows of a BCSC hardly ever are (a COO is listed by row).
template <bool BCSC>
int build_blocks(Coo c, std::uint32_t RW, const float* val, BlockArrays& out, std::uint32_t& B, Built& what,
                 hipStream_t st) {
    const bool tryGrouped = !BCSC && c.phases == 1;
    const std::uint64_t E = c.E;
    // ceil(length / 8) summed over at most min(RW, E) windows with edges
    const std::uint64_t maxB = std::min<std::uint64_t>(E, (E + 7 * std::min<std::uint64_t>(RW, E)) / 8);
    const bool exact = kBlockBytes * maxB > kCountFirst;
    const unsigned wBits = ceil_log2(RW);
    const bool places = BCSC && val;
    std::uint64_t *keysA = nullptr, *keysB = nullptr;
    std::uint32_t *winStart, *flags, *blocks, *scanTemp, *hist, *total;
    Lists L{};
    L.RW = RW;
    bool keys = !tryGrouped;
    // scratch, carved by the same function that sizes it; the partition's
    // part is a block of its own, taken where the COO is partitioned
    auto carve = [&](char* base, bool partition) {
        std::size_t off = 0;
        auto take = [&](std::size_t bytes) {
            char* p = base ? base + off : nullptr;
            off += align_up(bytes);
            return p;
        };
        if (partition) {
            keysA = reinterpret_cast<std::uint64_t*>(take(8 * E));
            keysB = reinterpret_cast<std::uint64_t*>(take(8 * E));
            hist = reinterpret_cast<std::uint32_t*>(take(4 * partition_hist_elems(E)));
            total = reinterpret_cast<std::uint32_t*>(take(4ull * kRadixBins));
            return off;
        }
        flags = reinterpret_cast<std::uint32_t*>(take(64));
        L.length = reinterpret_cast<std::uint32_t*>(take(4ull * RW + 64));
        winStart = reinterpret_cast<std::uint32_t*>(take(4ull * (RW + 1ull)));
        blocks = reinterpret_cast<std::uint32_t*>(take(RW > kOneScan || exact ? 4ull * (RW + 1ull) : 0));
        scanTemp = reinterpret_cast<std::uint32_t*>(take(RW > kOneScan ? 4 * scan_temp_elems(RW) : 0));
        L.mid = reinterpret_cast<std::uint32_t*>(take(4 * (E / kShort + 1)));
        L.big = reinterpret_cast<std::uint32_t*>(take(4 * (E / kMid + 1)));
        L.b = reinterpret_cast<std::uint32_t*>(take(4 * E));
        L.before = reinterpret_cast<std::uint32_t*>(take(4 * E));
        L.mask = reinterpret_cast<std::uint8_t*>(take(E));
        L.sPlace = places ? reinterpret_cast<std::uint32_t*>(take(4 * E)) : nullptr;
        L.sB = BCSC ? reinterpret_cast<std::uint32_t*>(take(4 * E)) : nullptr;
        L.sMask = BCSC ? reinterpret_cast<std::uint8_t*>(take(E)) : nullptr;
        L.winStart = winStart;
        L.flags = flags;
        return off;
    };
    L.longest = longest_window(E, c.numB);
    Scratch scratch, partition, byDegree;
    TCC_HIP_CHECK(scratch.take(carve(nullptr, false), st));
    carve(scratch.data(), false);
    // flags and list lengths lie together
    TCC_HIP_CHECK(fill<std::uint32_t>(flags, 64 + RW, 0u, st));
    const dim3 perEdge(grid_for(E, kThreads)), perEdge1(grid_for(E + 1, kThreads));
    if (tryGrouped) {
        hipLaunchKernelGGL(window_starts_kernel<false>, perEdge1, dim3(kThreads), 0, st, c, nullptr, RW, winStart, flags);
        TCC_LAUNCH_CHECK();
        TCC_HIP_CHECK(hipMemcpyAsync(scratch.mailHost(), flags, 8, hipMemcpyDeviceToHost, st));
        TCC_HIP_CHECK(scratch.wait());
        if (scratch.read()[kFlagRange]) {
            what = Built::Range;
            return TCC_OK;
        }
        keys = scratch.read()[kFlagUngrouped] != 0;
    }
    const std::uint64_t* grouped = nullptr;
    auto take_partition = [&]() -> int {
        if (partition.data()) return TCC_OK;
        TCC_HIP_CHECK(partition.take(carve(nullptr, true), st));
        carve(partition.data(), true);
        return TCC_OK;
    };
    if (keys) {
        // stable passes over the window's bits, the first from the COO
        if (const int rc = take_partition()) return rc;
        std::uint64_t* sorted = nullptr;
        TCC_HIP_CHECK(partition_by(CooLoad{c, flags}, keysA, keysB, E, c.bBits + 3, wBits, hist, total, &sorted, st));
        grouped = sorted;
        hipLaunchKernelGGL(window_starts_kernel<true>, perEdge1, dim3(kThreads), 0, st, c, grouped, RW, winStart, flags);
        TCC_LAUNCH_CHECK();
    }
    const dim3 listGrid(grid_for(RW, kListWaves)), listBlock(kListWaves * kWave);
    const dim3 otherGrid(static_cast<unsigned>(std::min<std::uint64_t>(E / kShort + 1, device_cus())));
    // KEYS: from the partitioned elements; else from the COO (BCSR only)
    auto lists = [&](auto fromKeys) {
        constexpr bool KEYS = decltype(fromKeys)::value;
        auto sorts = [&](auto keyType) {
            using K = decltype(keyType);
            hipLaunchKernelGGL((short_lists_kernel<KEYS, BCSC, K>), listGrid, listBlock, 0, st, c, grouped, L);
            if (E > kShort)
                hipLaunchKernelGGL((other_lists_kernel<KEYS, BCSC, K>), otherGrid, dim3(kLongThreads),
                                   other_lists_lds<K>(), st, c, grouped, L);
        };
        if (c.bBits <= 29) sorts(std::uint32_t{});  // b << 3 | a % 8, at most the ~0 of no edge, which sorts last
        else sorts(std::uint64_t{});
    };
    auto emit = [&](auto fromKeys) {
        constexpr bool KEYS = decltype(fromKeys)::value;
        hipLaunchKernelGGL((emit_blocks_kernel<KEYS, BCSC>), perEdge, dim3(kThreads), 0, st, c, grouped, L, out.off,
                           out.tcOffset, out.idx, out.bits, scratch.mail());
    };
    if constexpr (BCSC) {
        lists(std::true_type{});
    } else {
        if (keys) lists(std::true_type{});
        else lists(std::false_type{});
    }
    TCC_LAUNCH_CHECK();
    auto offsets = [&](std::uint32_t* off) -> int {
        if (RW <= kOneScan) {
            hipLaunchKernelGGL(window_blocks_kernel, dim3(1), dim3(1024), 0, st, L.length, RW, off);
        } else {
            hipLaunchKernelGGL(blocks_per_window_kernel, dim3(grid_for(RW, kThreads)), dim3(kThreads), 0, st, L.length,
                               RW, blocks);
            TCC_HIP_CHECK(exclusive_scan(blocks, off, RW, off + RW, scanTemp, st));
        }
        TCC_LAUNCH_CHECK();
        return TCC_OK;
    };
    auto read_mail = [&]() -> int {
        TCC_HIP_CHECK(scratch.wait());
        B = scratch.read()[0];
        what = scratch.read()[1] ? Built::Range : scratch.read()[2] ? Built::Duplicate
               : scratch.read()[3] ? Built::TooLong : Built::Ok;
        return TCC_OK;
    };
    // the blocks of the lists; the mail holds their count and the flags afterwards
    auto finish = [&]() -> int {
        if (exact) {
            if (const int rc = offsets(blocks)) return rc;
            hipLaunchKernelGGL(tell_host_kernel, dim3(1), dim3(1), 0, st, L, blocks, scratch.mail());
            TCC_LAUNCH_CHECK();
            if (const int rc = read_mail()) return rc;
            if (what != Built::Ok) return TCC_OK;
            TCC_HIP_CHECK(out.allocate(RW, B, E, val != nullptr));
            TCC_HIP_CHECK(hipMemcpyAsync(out.off, blocks, 4ull * (RW + 1ull), hipMemcpyDeviceToDevice, st));
        } else {
            if (!out.base) TCC_HIP_CHECK(out.allocate(RW, maxB, E, val != nullptr));
            if (const int rc = offsets(out.off)) return rc;
        }
        if constexpr (BCSC) {
            emit(std::true_type{});
        } else {
            if (keys) emit(std::true_type{});
            else emit(std::false_type{});
        }
        TCC_LAUNCH_CHECK();
        if (val) {
            hipLaunchKernelGGL(place_values_kernel<BCSC>, perEdge, dim3(kThreads), 0, st, c, L, out.off, out.tcOffset,
                               out.bits, val, out.data);
            TCC_LAUNCH_CHECK();
        }
        return read_mail();
    };
    // the lists again, of the whole COO sorted
    auto sort_all = [&]() -> int {
        if (const int rc = take_partition()) return rc;
        std::uint64_t* sorted = nullptr;
        TCC_HIP_CHECK(partition_by(CooLoad{c, flags}, keysA, keysB, E, 0, c.bBits + 3 + wBits, hist, total, &sorted, st));
        grouped = sorted;
        keys = true;
        // the entries before each edge, over the elements that the last pass read
        auto* pos = reinterpret_cast<std::uint32_t*>(sorted == keysA ? keysB : keysA);
        hipLaunchKernelGGL(entry_heads_kernel, perEdge, dim3(kThreads), 0, st, grouped, c.E, pos);
        TCC_LAUNCH_CHECK();
        TCC_HIP_CHECK(exclusive_scan(pos, pos, E, nullptr, pos + E, st));
        TCC_HIP_CHECK(fill<std::uint32_t>(flags + kFlagTooLong, 1, 0u, st));
        hipLaunchKernelGGL(sorted_lists_kernel<BCSC>, perEdge, dim3(kThreads), 0, st, grouped, pos, c.E, c.bBits, L);
        TCC_LAUNCH_CHECK();
        if constexpr (BCSC) {
            const std::size_t bytes = align_up(8 * E);
            TCC_HIP_CHECK(byDegree.take(2 * bytes, st));
            auto* elemsA = reinterpret_cast<std::uint64_t*>(byDegree.data());
            auto* elemsB = reinterpret_cast<std::uint64_t*>(byDegree.data() + bytes);
            hipLaunchKernelGGL(degree_elems_kernel, perEdge, dim3(kThreads), 0, st, grouped, c.E, c.bBits, L, elemsB);
            TCC_LAUNCH_CHECK();
            TCC_HIP_CHECK(partition_by(KeyLoad{elemsB, E}, elemsA, elemsB, E, 32, 3 + wBits, hist, total, &sorted, st));
            hipLaunchKernelGGL(degrees_kernel, perEdge, dim3(kThreads), 0, st, sorted, c.E, L, pos);
            TCC_LAUNCH_CHECK();
            TCC_HIP_CHECK(exclusive_scan(pos, pos, E, nullptr, pos + E, st));
            hipLaunchKernelGGL(degree_lists_kernel, perEdge, dim3(kThreads), 0, st, sorted, pos, c.E, L);
            TCC_LAUNCH_CHECK();
        }
        return TCC_OK;
    };
    int rc = finish();
    if (rc == TCC_OK && what == Built::TooLong) {
        rc = sort_all();
        if (rc == TCC_OK) rc = finish();
    }
    if (rc == TCC_OK && what == Built::Ok && !exact && kBlockBytes * (maxB - B) > kMaxSlack) {
        BlockArrays fit;
        if (fit.allocate(RW, B, E, val != nullptr) == hipSuccess) {
            const auto move = [&](void* to, const void* from, std::uint64_t bytes) {
                return bytes == 0 ? hipSuccess : hipMemcpyAsync(to, from, bytes, hipMemcpyDeviceToDevice, st);
            };
            if (move(fit.off, out.off, 4ull * (RW + 1ull)) == hipSuccess &&
                move(fit.tcOffset, out.tcOffset, 4ull * (B + 1ull)) == hipSuccess &&
                move(fit.idx, out.idx, 32ull * B) == hipSuccess && move(fit.bits, out.bits, 8ull * B) == hipSuccess &&
                move(fit.data, out.data, val ? 4 * E : 0) == hipSuccess && scratch.wait() == hipSuccess) {
                (void)pool_free(out.base);
                out = fit;
            } else {
                (void)pool_free(fit.base);
                set_last_error("HIP error while building the block arrays");
                rc = TCC_ERR_HIP;
            }
        } else {
            (void)hipGetLastError();  // no room for both: the larger ones stay
        }
    }
    if (rc == TCC_OK) {  // all work waited for, and none queued after it
        scratch.idle();
        partition.idle();
        byDegree.idle();
    }
    if (rc != TCC_OK || what != Built::Ok) {
        (void)hipStreamSynchronize(st);
        (void)pool_free(out.base);
        out.base = nullptr;
    }
    return rc;
}

int bcsc_by_conversion(const std::uint32_t* dRow, const std::uint32_t* dCol, const float* dVal, std::uint32_t nnz,
                       std::uint32_t numRows, std::uint32_t numCols, tcc_bcsc* out, void** allocation, hipStream_t st) {
    void* stream = st;
    tcc_swtcf_matrix m;
    tcc_swtcf_workspace ws;
    int rc = tcc_swtcf_alloc_matrix(&m, numRows, numCols, nnz, 1);
    if (rc) return rc;
    rc = tcc_swtcf_alloc_workspace(&ws, nnz, numCols, 1);
    if (rc) {
        tcc_swtcf_free_matrix(&m);
        return rc;
    }
    struct Cleanup {
        tcc_swtcf_matrix* m;
        tcc_swtcf_workspace* ws;
        ~Cleanup() {
            tcc_swtcf_free_workspace(ws);
            tcc_swtcf_free_matrix(m);
        }
    } cleanup{&m, &ws};
    rc = tcc_swtcf_convert(dRow, dCol, nnz, &m, &ws, stream);
    if (rc) return rc;
    const std::uint32_t CW = m.numColWindows;
    std::uint32_t hostErr = 0, T = 0, U = 0;
    TCC_HIP_CHECK(hipMemcpyAsync(&hostErr, ws.deviceError, 4, hipMemcpyDeviceToHost, st));
    TCC_HIP_CHECK(hipMemcpyAsync(&T, m.colWindowOffset + CW, 4, hipMemcpyDeviceToHost, st));
    TCC_HIP_CHECK(hipMemcpyAsync(&U, m.superWindowRowOffset + CW, 4, hipMemcpyDeviceToHost, st));
    TCC_HIP_CHECK(hipStreamSynchronize(st));
    TCC_REQUIRE(hostErr == 0, TCC_ERR_INVALID_ARGUMENT,
                "COO -> BCSC: converter error " + std::to_string(hostErr) + " (duplicates or indices out of range)");

    const std::size_t outBytes = align_up(4 * (CW + 1)) + align_up(4 * (T + 1)) + align_up(32 * std::max(T, 1u)) +
                                 align_up(8 * std::max(T, 1u)) + align_up(4 * nnz) + align_up(4 * std::max(U, 1u)) +
                                 align_up(4 * std::max(T, 1u)) + align_up(4 * scan_temp_elems(T + 1));
    char* o = nullptr;
    TCC_HIP_CHECK(device_malloc(&o, outBytes));
    char* q = o;
    auto takeOut = [&](std::size_t bytes) {
        char* p = q;
        q += align_up(bytes);
        return p;
    };
    auto* colWindowOffset = reinterpret_cast<std::uint32_t*>(takeOut(4 * (CW + 1)));
    auto* tcOffset = reinterpret_cast<std::uint32_t*>(takeOut(4 * (T + 1)));
    auto* sparseA2C = reinterpret_cast<std::uint32_t*>(takeOut(32 * std::max(T, 1u)));
    auto* tcLocalBit = reinterpret_cast<std::uint64_t*>(takeOut(8 * std::max(T, 1u)));
    auto* data = reinterpret_cast<float*>(takeOut(4 * nnz));
    auto* slotToLoc = reinterpret_cast<std::uint32_t*>(takeOut(4 * std::max(U, 1u)));  // scratch tail
    auto* counts = reinterpret_cast<std::uint32_t*>(takeOut(4 * std::max(T, 1u)));
    auto* temp = reinterpret_cast<std::uint32_t*>(takeOut(4 * scan_temp_elems(T + 1)));
    auto fail = [&](int code) {
        (void)hipFree(o);
        return code;
    };
    if (hipMemcpyAsync(colWindowOffset, m.colWindowOffset, 4 * (CW + 1), hipMemcpyDeviceToDevice, st) !=
            hipSuccess ||
        hipMemcpyAsync(tcLocalBit, m.tileLocalBit, 8ull * T, hipMemcpyDeviceToDevice, st) != hipSuccess) {
        set_last_error("HIP copy failed while building BCSC");
        return fail(TCC_ERR_HIP);
    }
    if (T > 0) {
        hipLaunchKernelGGL(bcsc_rows_kernel, dim3(grid_for(8ull * T, kThreads)), dim3(kThreads), 0, st,
                           m.colWindowOffset, CW, m.superWindowRowOffset, m.superWindowRows, m.tileRowSlot, T,
                           sparseA2C, slotToLoc);
        hipLaunchKernelGGL(popcount_kernel, dim3(grid_for(T, kThreads)), dim3(kThreads), 0, st, tcLocalBit, T,
                           counts);
    }
    if (exclusive_scan(counts, tcOffset, T, tcOffset + T, temp, st) != hipSuccess) return fail(TCC_ERR_HIP);
    hipLaunchKernelGGL(bcsc_values_kernel, dim3(grid_for(nnz, kThreads)), dim3(kThreads), 0, st, dRow, dCol, dVal,
                       nnz, m.superWindowRowOffset, m.superWindowRows, slotToLoc, tcLocalBit, tcOffset, data);
    if (hipGetLastError() != hipSuccess || hipStreamSynchronize(st) != hipSuccess) {
        set_last_error("HIP error while building BCSC");
        return fail(TCC_ERR_HIP);
    }
    out->num_rows = numRows;
    out->num_cols = numCols;
    out->nnz = nnz;
    out->num_TCBlocks = T;
    out->num_colWindows = CW;
    out->colWindowOffset = colWindowOffset;
    out->tcOffset = tcOffset;
    out->sparseA2C = sparseA2C;
    out->tcLocalBit = tcLocalBit;
    out->data = dVal ? data : nullptr;
    *allocation = o;
    return TCC_OK;
}

}  // namespace

extern "C" {

int tcc_block_release(void* allocation) {
    clear_last_error();
    if (allocation) TCC_HIP_CHECK(pool_free(allocation));
    return TCC_OK;
}

int tcc_coo_to_bcsr(const std::uint32_t* dRow, const std::uint32_t* dCol, const float* dVal, std::uint32_t nnz,
                    std::uint32_t numRows, std::uint32_t numCols, tcc_bcsr* out, void** allocation,
                    void* stream) {
    return tcc_coo_to_bcsr_phased(dRow, dCol, dVal, nnz, numRows, numCols, 1, out, allocation, stream);
}

int tcc_coo_to_bcsr_phased(const std::uint32_t* dRow, const std::uint32_t* dCol, const float* dVal,
                           std::uint32_t nnz, std::uint32_t numRows, std::uint32_t numCols, std::uint32_t phases,
                           tcc_bcsr* out, void** allocation, void* stream) {
    clear_last_error();
    TCC_REQUIRE(out && allocation && numRows >= 1 && numCols >= 1 && (nnz == 0 || (dRow && dCol)),
                TCC_ERR_INVALID_ARGUMENT, "invalid COO -> BCSR arguments");
    if (phases == 0) phases = 1;
    const hipStream_t st = as_stream(stream);
    const std::uint32_t windowsPerPhase = (numRows + 7) / 8;
    TCC_REQUIRE(static_cast<std::uint64_t>(windowsPerPhase) * phases < 0xFFFFFFFFull, TCC_ERR_UNSUPPORTED,
                "too many row windows for the phase count");
    const std::uint32_t RW = windowsPerPhase * phases;
    const unsigned colBits = std::max(1u, ceil_log2(numCols));
    TCC_REQUIRE(ceil_log2(RW) + colBits + 3 <= 64, TCC_ERR_UNSUPPORTED, "BCSR key exceeds 64 bits");
    std::memset(out, 0, sizeof(*out));
    *allocation = nullptr;
    BlockArrays arrays;
    std::uint32_t B = 0;
    if (nnz > 0) {
        const Coo c{dRow, dCol, nnz, numRows, numCols, phases, windowsPerPhase, colBits};
        Built what = Built::Ok;
        const int rc = build_blocks<false>(c, RW, dVal, arrays, B, what, st);
        if (rc) return rc;
        if (what != Built::Ok) {
            set_last_error(what == Built::Duplicate ? "duplicate (row, col) entries in the COO input"
                                                    : "COO index out of range");
            return TCC_ERR_INVALID_ARGUMENT;
        }
    } else {
        TCC_HIP_CHECK(arrays.allocate(RW, 0, 0, true));
        if (fill<std::uint32_t>(arrays.off, RW + 1ull, 0u, st) != hipSuccess ||
            fill<std::uint32_t>(arrays.tcOffset, 1, 0u, st) != hipSuccess || hipStreamSynchronize(st) != hipSuccess) {
            (void)pool_free(arrays.base);
            set_last_error("HIP error while building an empty BCSR");
            return TCC_ERR_HIP;
        }
    }
    out->num_rows = numRows;
    out->num_cols = numCols;
    out->nnz = nnz;
    out->num_TCBlocks = B;
    out->num_rowWindows = RW;
    out->rowWindowOffset = arrays.off;
    out->tcOffset = arrays.tcOffset;
    out->sparseA2B = arrays.idx;
    out->tcLocalBit = arrays.bits;
    out->data = dVal ? arrays.data : nullptr;
    out->phases = phases;
    *allocation = arrays.base;
    return TCC_OK;
}

int tcc_coo_to_bcsc(const std::uint32_t* dRow, const std::uint32_t* dCol, const float* dVal, std::uint32_t nnz,
                    std::uint32_t numRows, std::uint32_t numCols, tcc_bcsc* out, void** allocation,
                    void* stream) {
    clear_last_error();
    TCC_REQUIRE(out && allocation && numRows >= 1 && numCols >= 1 && (nnz == 0 || (dRow && dCol)),
                TCC_ERR_INVALID_ARGUMENT, "invalid COO -> BCSC arguments");
    const hipStream_t st = as_stream(stream);
    std::memset(out, 0, sizeof(*out));
    *allocation = nullptr;
    if (nnz == 0) {
        // every column window empty and no blocks, as tcc_coo_to_bcsr gives
        // for no edges (the converter below needs at least one edge)
        const std::uint32_t CW = (numCols + 7) / 8;
        const std::size_t offBytes = align_up(4ull * (CW + 1));
        char* o = nullptr;
        TCC_HIP_CHECK(device_malloc(&o, offBytes + align_up(4) + align_up(32) + align_up(8)));
        if (fill<std::uint32_t>(reinterpret_cast<std::uint32_t*>(o), (offBytes + align_up(4) + align_up(32) + align_up(8)) / 4,
                                0u, st) != hipSuccess ||
            hipStreamSynchronize(st) != hipSuccess) {
            (void)hipFree(o);
            set_last_error("HIP error while building an empty BCSC");
            return TCC_ERR_HIP;
        }
        out->num_rows = numRows;
        out->num_cols = numCols;
        out->num_colWindows = CW;
        out->colWindowOffset = reinterpret_cast<std::uint32_t*>(o);
        out->tcOffset = reinterpret_cast<std::uint32_t*>(o + offBytes);
        out->sparseA2C = reinterpret_cast<std::uint32_t*>(o + offBytes + align_up(4));
        out->tcLocalBit = reinterpret_cast<std::uint64_t*>(o + offBytes + align_up(4) + align_up(32));
        *allocation = o;
        return TCC_OK;
    }
    BlockArrays arrays;
    std::uint32_t B = 0;
    Built what = Built::Ok;
    const std::uint32_t CW = (numCols + 7) / 8;
    const unsigned rowBits = std::max(1u, ceil_log2(numRows));
    if (ceil_log2(CW) + rowBits + 3 <= 64) {
        const Coo c{dCol, dRow, nnz, numCols, numRows, 1, CW, rowBits};
        const int rc = build_blocks<true>(c, CW, dVal, arrays, B, what, st);
        if (rc) return rc;
    } else {
        what = Built::Range;
    }
    if (what != Built::Ok) return bcsc_by_conversion(dRow, dCol, dVal, nnz, numRows, numCols, out, allocation, st);
    out->num_rows = numRows;
    out->num_cols = numCols;
    out->nnz = nnz;
    out->num_TCBlocks = B;
    out->num_colWindows = CW;
    out->colWindowOffset = arrays.off;
    out->tcOffset = arrays.tcOffset;
    out->sparseA2C = arrays.idx;
    out->tcLocalBit = arrays.bits;
    out->data = dVal ? arrays.data : nullptr;
    *allocation = arrays.base;
    return TCC_OK;
}

}  // extern "C"
