// Id -> slot map of one partition's ghosts: home slot and launchers
// (hashmap.hip).  Layout and probing of the reference's GPUHashMap
// (gpu_kernels.py:91-260).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define SS_MAP_INSERT 0
#define SS_MAP_REMOVE 1
#define SS_MAP_RAW 2

// floor-mod of the wrapped int64 product id * 2654435761 by the capacity, as
// the reference's numpy expression computes it (gpu_kernels.py:112-114, :146)
__host__ __device__ __forceinline__ int64_t ss_map_home(int64_t id, int64_t cap) {
    const int64_t h = (int64_t)((uint64_t)id * 2654435761ull);
    int64_t s = h % cap;
    return s < 0 ? s + cap : s;
}

// keys = -1, values = -1 over the whole table
hipError_t ss_launch_map_clear(unsigned long long *keys, int32_t *vals, int64_t cap, hipStream_t s);
// *bad = 1 when an id is reserved or a slot outside [0, n_total)
hipError_t ss_launch_map_check(const int64_t *ids, const int32_t *slots, int64_t n, int64_t n_total, uint32_t *bad,
                               hipStream_t s);
// build of n < cap entries into the whole table; claim: workspace of cap words
hipError_t ss_launch_map_build(unsigned long long *keys, int32_t *vals, int64_t cap, const int64_t *ids,
                               const int32_t *slot_vals, int64_t n, unsigned long long *claim, int num_cus,
                               hipStream_t s);
// insert / remove / raw re-insert of n entries in input order; out[0] +=
// entries added or removed, out[1] += entries that found no slot
hipError_t ss_launch_map_seq(unsigned long long *keys, int32_t *vals, int64_t cap, int op, const int64_t *ids,
                             const int32_t *slot_vals, int64_t n, int32_t *out, hipStream_t s);
