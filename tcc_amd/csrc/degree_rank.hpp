// Degree ranks of the rows or columns of a COO matrix, for the
// degree-sorted formats (row super-window BCSR, dense hub tiles): rank[i] is
// the position of index i when the indices are ordered by degree
// (descending) and then by index (ascending).
#pragma once

#include "common.hpp"
#include "primitives.hpp"

namespace tcc {
namespace {

__global__ void degree_kernel(const std::uint32_t* __restrict__ idx, std::uint32_t E, std::uint32_t limit,
                              std::uint32_t* __restrict__ deg, std::uint32_t* __restrict__ err) {
    const std::uint32_t e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= E) return;
    const std::uint32_t v = idx[e];
    if (v >= limit) {
        atomicMax(err, 1u);
        return;
    }
    atomicAdd(&deg[v], 1u);
}

// Degrees counted in LDS: workgroup b takes slice b % slices of 32K indices
// and a share of the edges, counts the edges of its slice there and adds its
// counts to deg at the end, consecutive indices together.  An atomic per edge
// on deg itself queues on the hubs (one address takes about 12 ns an add: 4.4
// ms for 57M edges of a skewed 233k-node graph, whose top row has 0.4M of
// them; 0.2 ms this way).  The edges are read once per slice, so past
// kDegreeSlices of them the atomics are left.
constexpr std::uint32_t kDegreeSlice = 32768;
constexpr std::uint32_t kDegreeSlices = 16;
__global__ void __launch_bounds__(1024) degree_slices_kernel(const std::uint32_t* __restrict__ idx, std::uint32_t E,
                                                            std::uint32_t limit, std::uint32_t slices,
                                                            std::uint32_t perShare, std::uint32_t* __restrict__ deg,
                                                            std::uint32_t* __restrict__ err) {
    extern __shared__ std::uint32_t counts[];  // [kDegreeSlice]
    for (unsigned i = threadIdx.x; i < kDegreeSlice; i += 1024) counts[i] = 0;
    __syncthreads();
    const std::uint32_t slice = blockIdx.x % slices;
    const std::uint64_t begin = static_cast<std::uint64_t>(blockIdx.x / slices) * perShare;
    const std::uint64_t end = begin + perShare < E ? begin + perShare : E;
    const std::uint32_t base = slice * kDegreeSlice;
    bool bad = false;
    auto count = [&](std::uint32_t v, bool valid) {
        bad |= valid && v >= limit;
        const std::uint32_t x = v - base;  // wraps below the slice
        const bool mine = valid && x < kDegreeSlice && v < limit;
        // the lanes that share the first such lane's index (a COO listed by
        // row has runs of one) add together
        const std::uint64_t todo = __ballot(mine);
        if (todo == 0) return;
        const std::uint32_t lead = static_cast<std::uint32_t>(
            __builtin_amdgcn_readlane(static_cast<int>(x), __builtin_ctzll(todo)));
        const std::uint64_t same = __ballot(mine && x == lead);
        if (mine && x != lead) atomicAdd(&counts[x], 1u);
        if (__lane_id() == static_cast<unsigned>(__builtin_ctzll(todo)))
            atomicAdd(&counts[lead], static_cast<std::uint32_t>(__popcll(same)));
    };
    // shares are multiples of 4 edges: 16 edges a thread and step in four
    // 16-byte loads where idx is aligned for them
    if ((reinterpret_cast<std::uintptr_t>(idx) & 15u) == 0) {
        const std::uint64_t whole = end & ~3ull;
        for (std::uint64_t e1 = begin; e1 < whole; e1 += 16 * 1024) {
            vu4 v[4];
#pragma unroll
            for (unsigned q = 0; q < 4; ++q) {
                const std::uint64_t i = e1 + 4 * (q * 1024 + threadIdx.x);
                v[q] = load_global<vu4>(idx + (i < whole ? i : whole - 4));
            }
#pragma unroll
            for (unsigned q = 0; q < 4; ++q) {
                const bool valid = e1 + 4 * (q * 1024 + threadIdx.x) < whole;
                count(v[q].x, valid);
                count(v[q].y, valid);
                count(v[q].z, valid);
                count(v[q].w, valid);
            }
        }
        const std::uint64_t i = whole + threadIdx.x;
        if (whole < end) count(idx[i < end ? i : end - 1], i < end);
    } else {
        for (std::uint64_t e1 = begin; e1 < end; e1 += 1024) {
            const std::uint64_t i = e1 + threadIdx.x;
            count(idx[i < end ? i : end - 1], i < end);
        }
    }
    raise_flag(err, bad);
    __syncthreads();
    for (unsigned i = threadIdx.x; i < kDegreeSlice; i += 1024)
        if (counts[i]) atomicAdd(&deg[base + i], counts[i]);
}

// key = (~deg << idBits) | id: ascending order = degree descending, ids ascending.
__global__ void degree_keys_kernel(const std::uint32_t* __restrict__ deg, std::uint32_t n, unsigned idBits,
                                   std::uint64_t* __restrict__ keys) {
    const std::uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) keys[i] = (static_cast<std::uint64_t>(0xFFFFFFFFu - deg[i]) << idBits) | i;
}

// order[s] = id at sorted position s (0xFFFFFFFF for s in [n, padded)),
// rank[id] = s.  `order` may be null.
__global__ void order_rank_kernel(const std::uint64_t* __restrict__ sorted, std::uint32_t n, std::uint32_t padded,
                                  unsigned idBits, std::uint32_t* __restrict__ order, std::uint32_t* __restrict__ rank) {
    const std::uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= padded) return;
    if (s >= n) {
        if (order) order[s] = 0xFFFFFFFFu;
        return;
    }
    const std::uint32_t id = static_cast<std::uint32_t>(sorted[s] & ((1ull << idBits) - 1ull));
    if (order) order[s] = id;
    rank[id] = s;
}

inline unsigned rank_bits(std::uint64_t x) {
    unsigned b = 0;
    while ((1ull << b) < x) ++b;
    return b;
}

// deg[0..limit) += occurrences of each index in idx[0..E); indices >= limit
// set *err to 1.  deg must be zeroed by the caller.
inline hipError_t degree_histogram(const std::uint32_t* idx, std::uint32_t E, std::uint32_t limit,
                                   std::uint32_t* deg, std::uint32_t* err, hipStream_t st) {
    if (E == 0) return hipSuccess;
    const std::uint32_t slices = limit / kDegreeSlice + (limit % kDegreeSlice != 0);
    if (slices <= kDegreeSlices) {
        // about one workgroup per compute unit (its LDS holds one), 64K edges at least
        const std::uint32_t shares = static_cast<std::uint32_t>(
            std::min<std::uint64_t>(std::max(1u, device_cus() / slices), (E + 65535ull) / 65536));
        const std::uint32_t per =
            static_cast<std::uint32_t>(std::min<std::uint64_t>((static_cast<std::uint64_t>(E) + shares - 1) / shares + 3, 0xFFFFFFFCull)) & ~3u;
        hipLaunchKernelGGL(degree_slices_kernel, dim3(slices * shares), dim3(1024), 4 * kDegreeSlice, st, idx, E, limit,
                           slices, per, deg, err);
    } else {
        hipLaunchKernelGGL(degree_kernel, dim3(grid_for(E, 256)), dim3(256), 0, st, idx, E, limit, deg, err);
    }
    return hipGetLastError();
}

// rank[] and (optionally) order[] of n indices with degrees deg[] of at most
// maxDegree; keysA, keysB hold n u64 each, temp radix_temp_elems(n) u32.
// The ids are in order to begin with, so stable passes over the degree's
// bits alone give the order.
inline hipError_t degree_ranks(const std::uint32_t* deg, std::uint32_t n, std::uint32_t maxDegree, std::uint32_t padded,
                               std::uint32_t* rank,
                               std::uint32_t* order, std::uint64_t* keysA, std::uint64_t* keysB, std::uint32_t* temp,
                               hipStream_t st) {
    const unsigned idBits = std::max(1u, rank_bits(n));
    hipLaunchKernelGGL(degree_keys_kernel, dim3(grid_for(n, 256)), dim3(256), 0, st, deg, n, idBits, keysB);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    std::uint64_t* sorted = nullptr;
    e = partition_by(KeyLoad{keysB, n}, keysA, keysB, n, idBits, rank_bits(static_cast<std::uint64_t>(maxDegree) + 1),
                     temp, temp + partition_hist_elems(n), &sorted, st);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(order_rank_kernel, dim3(grid_for(padded, 256)), dim3(256), 0, st, sorted, n, padded, idBits,
                       order, rank);
    return hipGetLastError();
}

}  // namespace
}  // namespace tcc
