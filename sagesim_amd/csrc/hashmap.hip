// Open-addressing id -> slot map of one partition's ghosts, laid out as the
// reference's GPUHashMap (gpu_kernels.py:91-260): keys int64 (-1 empty,
// -2 deleted), values int32 (-1 in empty and deleted slots), home slot the
// floor-mod of the wrapped int64 product id * 2654435761 by the capacity
// (gpu_kernels.py:112-114, :146), linear probing.  Every operation leaves the
// arrays exactly as the reference's CPU mirror would be after the same calls:
//   * build (gpu_kernels.py:122-169) places entries in rounds: in every round
//     the remaining entry of lowest input index among those probing an empty
//     slot takes it, all others advance one slot.  So a slot goes to the entry
//     that reaches it after the fewest steps, the lowest index among equals, and
//     every entry takes the first slot that would have it: the stable matching
//     of entries (which prefer nearer slots) and slots (which prefer (steps,
//     index)), which proposals reach in any order when a slot may change its
//     mind.  One launch does it, with no rounds and no counts read back;
//   * insert, remove (gpu_kernels.py:171-206) and the re-insertion of a
//     resize (gpu_kernels.py:221-247) are sequential in the reference, and one
//     entry's probe depends on the writes of the entries before it, so they
//     run in input order on one wavefront, 64 slots of the probe per load.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "ss_map.h"

namespace {

constexpr unsigned long long kEmpty = (unsigned long long)(-1ll);
constexpr unsigned long long kDeleted = (unsigned long long)(-2ll);

__global__ void map_fill_kernel(unsigned long long *keys, int32_t *vals, int64_t cap) {
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g < cap) {
        keys[g] = kEmpty;
        vals[g] = -1;
    }
}

// *bad = 1 (page-locked) when an id is reserved (-1, -2) or a slot outside [0, n_total)
__global__ __launch_bounds__(256) void map_check_kernel(const int64_t *__restrict__ ids,
                                                        const int32_t *__restrict__ slots, int64_t n, uint32_t n_total,
                                                        uint32_t *bad) {
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= n) return;
    const int64_t id = ids[g];
    if (id == -1 || id == -2 || (uint32_t)slots[g] >= n_total) *bad = 1u;
}

// ---- build ----
// claim[s] = steps << 32 | index of the entry that holds slot s (all ones:
// none).  A thread carries one entry at a time to its next slot until a slot
// takes it for good, going on with the entry it displaces, if any; claims only
// fall and every step moves an entry one slot on, so all end (n < cap).  Bound
// by the 64-bit atomics, one random line each, 1.5 an entry at load 0.5: 1.6M
// entries in 104 us and 54 us for the table (the rounds: 44 of 19 us and 11
// synchronisations, 3.9 ms of a build with its allocations, now 1.6).
__global__ __launch_bounds__(256) void map_bid_kernel(const int64_t *__restrict__ ids, int64_t n, int64_t cap,
                                                      unsigned long long *claim) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; g < n; g += stride) {
        unsigned long long mine = (unsigned long long)g;
        int64_t s = ss_map_home(ids[g], cap);
        for (;;) {
            const unsigned long long old = atomicMin(&claim[s], mine);
            if (old == kEmpty) break;
            if (old > mine) mine = old;                 // displaced: goes on from here
            mine += 1ull << 32;
            s = s + 1 == cap ? 0 : s + 1;
        }
    }
}

// the table from its claims (empty slots: key and value -1)
__global__ __launch_bounds__(256) void map_place_kernel(const unsigned long long *__restrict__ claim, int64_t cap,
                                                        const int64_t *__restrict__ ids,
                                                        const int32_t *__restrict__ slot_vals,
                                                        unsigned long long *__restrict__ keys, int32_t *__restrict__ vals) {
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= cap) return;
    const unsigned long long c = claim[s];
    const uint32_t i = (uint32_t)c;
    keys[s] = c == kEmpty ? kEmpty : (unsigned long long)ids[i];
    vals[s] = c == kEmpty ? -1 : slot_vals[i];
}

__global__ __launch_bounds__(256) void map_unclaim_kernel(unsigned long long *claim, int64_t cap) {
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (s < cap) claim[s] = kEmpty;
}

// ---- sequential operations on one wavefront ----
// op SS_MAP_INSERT: stop at an empty or deleted slot or at the id's own key
//    (gpu_kernels.py:175-179); a slot that does not hold the id yet counts as
//    a new entry (:181-182); key and value are written.
// op SS_MAP_REMOVE: stop at an empty slot (not found) or at the id's key,
//    which becomes deleted with value -1 (gpu_kernels.py:193-206).
// op SS_MAP_RAW: stop at an empty or deleted slot (gpu_kernels.py:242-247).
// out[0] += entries added (insert, raw) or removed (remove); out[1] += ops
// that found no stop slot within one sweep of the table (a full table; the
// reference would probe forever).
__global__ __launch_bounds__(64) void map_seq_kernel(unsigned long long *keys, int32_t *vals, int64_t cap, int op,
                                                     const int64_t *__restrict__ ids,
                                                     const int32_t *__restrict__ slot_vals, int64_t n, int32_t *out) {
    const int lane = threadIdx.x;
    int32_t changed = 0, failed = 0;
    for (int64_t i = 0; i < n; ++i) {
        const int64_t id = ids[i];
        const unsigned long long key = (unsigned long long)id;
        int64_t base = ss_map_home(id, cap);
        int64_t stop = -1;
        for (int64_t swept = 0; swept < cap; swept += 64) {
            int64_t s = base + lane;
            if (s >= cap) s -= cap;            // base < cap and lane < 64 <= cap
            const unsigned long long k = keys[s];
            bool hit;
            if (op == SS_MAP_INSERT) hit = k == kEmpty || k == kDeleted || k == key;
            else if (op == SS_MAP_REMOVE) hit = k == kEmpty || k == key;
            else hit = k == kEmpty || k == kDeleted;
            // slots past one whole sweep of the table do not count
            hit = hit && swept + lane < cap;
            const unsigned long long b = __ballot(hit);
            if (b) {
                const int f = __ffsll((long long)b) - 1;
                stop = __shfl(s, f);
                break;
            }
            base += 64;
            if (base >= cap) base -= cap;
        }
        if (stop < 0) {
            ++failed;
        } else if (lane == 0) {
            const unsigned long long k = keys[stop];
            if (op == SS_MAP_REMOVE) {
                if (k == key) {
                    keys[stop] = kDeleted;
                    vals[stop] = -1;
                    ++changed;
                }
            } else {
                if (op == SS_MAP_RAW || k != key) ++changed;
                keys[stop] = key;
                vals[stop] = slot_vals[i];
            }
        }
        // the next entry's probe must see this entry's write: wait for the
        // store and drop this CU's cached lines of the table
        __threadfence();
    }
    if (lane == 0) {
        out[0] += changed;
        out[1] += failed;
    }
}

inline unsigned grid_of(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

}  // namespace

hipError_t ss_launch_map_clear(unsigned long long *keys, int32_t *vals, int64_t cap, hipStream_t s) {
    if (cap <= 0) return hipSuccess;
    hipLaunchKernelGGL(map_fill_kernel, dim3(grid_of(cap, 256)), dim3(256), 0, s, keys, vals, cap);
    return hipGetLastError();
}

hipError_t ss_launch_map_check(const int64_t *ids, const int32_t *slots, int64_t n, int64_t n_total, uint32_t *bad,
                               hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(map_check_kernel, dim3(grid_of(n, 256)), dim3(256), 0, s, ids, slots, n, (uint32_t)n_total, bad);
    return hipGetLastError();
}

hipError_t ss_launch_map_build(unsigned long long *keys, int32_t *vals, int64_t cap, const int64_t *ids,
                               const int32_t *slot_vals, int64_t n, unsigned long long *claim, int num_cus,
                               hipStream_t s) {
    if (cap <= 0) return hipSuccess;
    hipLaunchKernelGGL(map_unclaim_kernel, dim3(grid_of(cap, 256)), dim3(256), 0, s, claim, cap);
    if (n > 0) {
        const unsigned g = grid_of(n, 256), most = (unsigned)num_cus * 8u;
        hipLaunchKernelGGL(map_bid_kernel, dim3(g < most ? g : most), dim3(256), 0, s, ids, n, cap, claim);
    }
    hipLaunchKernelGGL(map_place_kernel, dim3(grid_of(cap, 256)), dim3(256), 0, s, claim, cap, ids, slot_vals, keys,
                       vals);
    return hipGetLastError();
}

hipError_t ss_launch_map_seq(unsigned long long *keys, int32_t *vals, int64_t cap, int op, const int64_t *ids,
                             const int32_t *slot_vals, int64_t n, int32_t *out, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(map_seq_kernel, dim3(1), dim3(64), 0, s, keys, vals, cap, op, ids, slot_vals, n, out);
    return hipGetLastError();
}
