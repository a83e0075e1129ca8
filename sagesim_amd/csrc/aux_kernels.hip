// Kernels around the tick: CSR symmetry check, bitmap rebuilds, id -> slot
// lookups in the ghost map, the halo refresh and packing, census, and the
// two probes the measurement uses (a streaming copy and a random gather).
// The tick kernel itself and its direction-state kernels are in
// tick_kernels.hip.
#include <algorithm>

#include "ss_device.h"
#include "ss_runtime.h"

namespace {

// 64-bit finaliser of splitmix64 (Steele, Lea, Flood 2014).
__device__ __forceinline__ uint64_t mix64(uint64_t x) {
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}

// Symmetry of a CSR as a multiset test: the sums of two independent hashes
// over all entries (i, j) equal those over the mirrored entries (j, i) when
// every entry has its mirror.
// Row b of part (SS_STATS_ROW words, page-locked) gets block b's words 0 .. 3:
// the sums, and 4: the complement of the first entry outside [0, n_total), 0 if
// all are inside.  A thread takes 16 entries at a time (64 bytes) wherever its rows begin,
// and finds the row of the first by halving, so that a hub's row is shared by as
// many threads as it has entries for.  Bound by the 64-bit products (eight an
// entry) and the halving's chain of loads, once for 16 entries: 36 us for the
// 6.8M entries of a BA(851k), where a row to a thread took 1033 us, the longest
// row's walk.  Rows that do not ascend only give sums that nobody uses.
__device__ __forceinline__ int64_t row_of(const int64_t *__restrict__ row_ptr, int64_t j, int64_t lo, int64_t hi) {
    while (hi - lo > 1) {                               // the last row in [lo, hi) that begins at or before j
        const int64_t mid = (lo + hi) >> 1;
        if (row_ptr[mid] <= j) lo = mid;
        else hi = mid;
    }
    return lo;
}

__global__ __launch_bounds__(256) void entries_kernel(const int64_t *__restrict__ row_ptr,
                                                      const int32_t *__restrict__ col, int64_t n, int64_t nnz,
                                                      int64_t n_total, unsigned long long *part) {
    unsigned long long h[5] = {0, 0, 0, 0, 0};
    const int64_t stride = 16 * (int64_t)gridDim.x * blockDim.x;
    for (int64_t j0 = 16 * ((int64_t)blockIdx.x * blockDim.x + threadIdx.x); j0 < nnz; j0 += stride) {
        int64_t i = row_of(row_ptr, j0, 0, n), next = row_ptr[i + 1];
        auto entry = [&](int64_t j, int32_t e) {
            if (j >= next && i + 1 < n) {
                next = row_ptr[++i + 1];
                if (j >= next) {                        // past empty rows
                    i = row_of(row_ptr, j, i, n);
                    next = row_ptr[i + 1];
                }
            }
            if ((e < 0 || (int64_t)e >= n_total) && ~(unsigned long long)j > h[4]) h[4] = ~(unsigned long long)j;
            const uint64_t c = (uint32_t)e;
            const uint64_t fwd = ((uint64_t)i << 32) | c, bwd = (c << 32) | (uint64_t)i;
            h[0] += mix64(fwd ^ 0x9E3779B97F4A7C15ull);
            h[1] += mix64(fwd * 0xD6E8FEB86659FD93ull + 0x2545F4914F6CDD1Dull);
            h[2] += mix64(bwd ^ 0x9E3779B97F4A7C15ull);
            h[3] += mix64(bwd * 0xD6E8FEB86659FD93ull + 0x2545F4914F6CDD1Dull);
        };
        if (j0 + 16 <= nnz) {
            int4 v[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) v[q] = *(const int4 *)(col + j0 + 4 * q);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                entry(j0 + 4 * q, v[q].x);
                entry(j0 + 4 * q + 1, v[q].y);
                entry(j0 + 4 * q + 2, v[q].z);
                entry(j0 + 4 * q + 3, v[q].w);
            }
        } else {
            for (int64_t j = j0; j < nnz; ++j) entry(j, col[j]);
        }
    }
    __shared__ unsigned long long red[4][5];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
#pragma unroll
        for (int q = 0; q < 4; ++q) h[q] += __shfl_down(h[q], off);
        const unsigned long long o = __shfl_down(h[4], off);
        h[4] = o > h[4] ? o : h[4];
    }
    if ((threadIdx.x & 63) == 0)
        for (int q = 0; q < 5; ++q) red[threadIdx.x >> 6][q] = h[q];
    __syncthreads();
    if (threadIdx.x < 5) {
        unsigned long long t = red[0][threadIdx.x];
        for (int w = 1; w < 4; ++w) {
            const unsigned long long o = red[w][threadIdx.x];
            t = threadIdx.x < 4 ? t + o : o > t ? o : t;
        }
        part[SS_STATS_ROW * blockIdx.x + threadIdx.x] = t;
    }
}

// What a replica keeps by agent, from its rows and key ids, in one pass: degrees
// in a byte, the key ids' low words, the entries before every 64th agent, the
// empty rows of the ghosts (nnz each).  Row b of part gets words 5: the
// complement of the first row that is negative (0: none), 6: the longest row,
// 7: the high words of the key ids or'ed.  Bound by the 21 bytes an agent.
__global__ __launch_bounds__(256) void agents_kernel(int64_t *__restrict__ row_ptr, const int64_t *__restrict__ ids,
                                                     int64_t n, int64_t n_total, int64_t nnz, uint8_t *__restrict__ deg8,
                                                     uint32_t *__restrict__ lo, int64_t *__restrict__ edge64,
                                                     unsigned long long *part) {
    unsigned long long w[3] = {0, 0, 0};
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i <= n_total; i += stride) {
        const int64_t b = i <= n && n > 0 ? row_ptr[i] : nnz;
        if (i > n || n == 0) row_ptr[i] = nnz;
        if (i % 64 == 0 && i < n_total) edge64[i / 64] = b;
        if (i >= n) continue;
        const int64_t d = row_ptr[i + 1] - b;
        deg8[i] = (uint8_t)(d < 0 ? 0 : d < 255 ? d : 255);
        if (d < 0) w[0] = ~(unsigned long long)i > w[0] ? ~(unsigned long long)i : w[0];
        else w[1] = (unsigned long long)d > w[1] ? (unsigned long long)d : w[1];
        const uint64_t id = (uint64_t)ids[i];
        lo[i] = (uint32_t)id;
        w[2] |= id >> 32;
    }
    __shared__ unsigned long long red[4][3];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const unsigned long long o = __shfl_down(w[q], off);
            w[q] = q == 2 ? w[q] | o : o > w[q] ? o : w[q];
        }
    if ((threadIdx.x & 63) == 0)
        for (int q = 0; q < 3; ++q) red[threadIdx.x >> 6][q] = w[q];
    __syncthreads();
    if (threadIdx.x < 3) {
        unsigned long long t = red[0][threadIdx.x];
        for (int v = 1; v < 4; ++v) {
            const unsigned long long o = red[v][threadIdx.x];
            t = threadIdx.x == 2 ? t | o : o > t ? o : t;
        }
        part[SS_STATS_ROW * blockIdx.x + 5 + threadIdx.x] = t;
    }
}

__global__ __launch_bounds__(256) void high_words_kernel(const int64_t *__restrict__ ids, int64_t n,
                                                         uint32_t *__restrict__ hi) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) hi[i] = (uint32_t)((uint64_t)ids[i] >> 32);
}

// Rebuild bitmap words [w0, w1) of one state buffer.
__global__ void bits_kernel(const int8_t *__restrict__ st, uint64_t *__restrict__ bits, int64_t w0,
                            int64_t w1, int64_t n_total, int8_t inf) {
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t i = w0 * 64 + g;
    const bool on = i < w1 * 64 && i < n_total && st[i] == inf;
    const uint64_t word = __ballot(on);
    if ((threadIdx.x & 63) == 0 && (i >> 6) < w1) bits[i >> 6] = word;
}

// ---- id -> slot lookups (gpu_kernels.py:208-215): probe from the home slot
// until the id or an empty slot ----
__device__ __forceinline__ int32_t map_find(const unsigned long long *__restrict__ keys,
                                            const int32_t *__restrict__ vals, int64_t cap, int64_t id) {
    int64_t s = ss_map_home(id, cap);
    for (int64_t probe = 0; probe < cap; ++probe) {
        const unsigned long long k = keys[s];
        if (k == (unsigned long long)id) return vals[s];
        if (k == (unsigned long long)(-1ll)) return -1;
        s = s + 1 == cap ? 0 : s + 1;
    }
    return -1;
}

// counts[0] += lookups that found nothing, counts[1] = min of the slots found
// (as unsigned words; LOWEST only).  One atomic per block and count: they run
// one after another.
template <bool LOWEST>
__global__ __launch_bounds__(256) void map_lookup_kernel(const unsigned long long *__restrict__ keys,
                                                         const int32_t *__restrict__ vals, int64_t cap,
                                                         const int64_t *__restrict__ ids, int32_t *__restrict__ out,
                                                         int64_t n, uint32_t *counts) {
    __shared__ uint32_t miss, low;
    if (threadIdx.x == 0) {
        miss = 0u;
        low = ~0u;
    }
    __syncthreads();
    uint32_t m = 0u, lo = ~0u;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; g < n; g += stride) {
        const int32_t v = map_find(keys, vals, cap, ids[g]);
        out[g] = v;
        if (v < 0) ++m;
        else if ((uint32_t)v < lo) lo = (uint32_t)v;
    }
    if (m) atomicAdd(&miss, m);
    if (LOWEST && lo != ~0u) atomicMin(&low, lo);
    __syncthreads();
    if (threadIdx.x == 0) {
        if (miss) atomicAdd(&counts[0], miss);
        if (LOWEST && low != ~0u) atomicMin(&counts[1], low);
    }
}

// rec[slot[h] - base] = the last record h of every slot (rec cleared to -1)
__global__ __launch_bounds__(256) void halo_records_kernel(const int32_t *__restrict__ slot, int64_t n, int64_t base,
                                                           int32_t *rec) {
    const int64_t h = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (h < n && slot[h] >= 0) atomicMax(&rec[slot[h] - base], (int32_t)h);
}

__global__ void fill_i32_kernel(int32_t *p, int64_t n, int32_t v) {
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g < n) p[g] = v;
}

// Ghost refresh (gpu_kernels.py:1030-1036 writes ghosts into the read and the
// write buffer): record h of the halo goes to slot slots[h].
// Ghost refresh in slot order: slot base + g takes record rec[g] of the halo
// (-1: not bound, state kept) into both state buffers, and the bitmap words
// of the slots [base, n_total) are rebuilt from the states of the buffer the
// next tick reads (`cur`, `bits`).  base is a multiple of 64.  One gather per
// slot and whole-word writes, where a scatter in record order would write
// single bytes all over the slots.
// PACKED: the halo holds 2-bit state codes, record h in bits 2 (h % 4) and
// 2 (h % 4) + 1 of byte h / 4.
template <bool PACKED>
__global__ void halo_gather_kernel(int8_t *s0, int8_t *s1, const int8_t *cur, uint64_t *__restrict__ bits,
                                   const int32_t *__restrict__ rec, const int8_t *__restrict__ vals, int64_t base,
                                   int64_t n_total, int8_t inf) {
    // four slots per thread (base is a multiple of 64, the record list is
    // padded to whole groups of four with -1): one 16-byte record load, four
    // value reads, one 4-byte store per state buffer; a wavefront covers 256
    // slots, four bitmap words
    const int lane = threadIdx.x & 63;
    const int64_t i = base + 4 * ((int64_t)blockIdx.x * blockDim.x + threadIdx.x);
    uint32_t nib = 0u;                                   // infectious bits of the four slots
    if (i < n_total) {
        const int4 h = *(const int4 *)(rec + (i - base));
        const int32_t hh[4] = {h.x, h.y, h.z, h.w};
        uint32_t v4 = 0u;
        bool any_rec = false, all_rec = true;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            any_rec |= hh[q] >= 0;
            all_rec &= hh[q] >= 0;
        }
        if (!all_rec) {
            // slots without a record keep their state; a whole group in range
            // reads it as one word
            if (i + 3 < n_total) {
                v4 = *(const uint32_t *)(cur + i);
            } else {
                for (int q = 0; q < 4 && i + q < n_total; ++q) v4 |= (uint32_t)(uint8_t)cur[i + q] << (8 * q);
            }
        }
        if (any_rec) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (hh[q] >= 0) {
                    uint32_t v;
                    if constexpr (PACKED)
                        v = ((uint32_t)(uint8_t)vals[hh[q] >> 2] >> ((hh[q] & 3) * 2)) & 3u;
                    else
                        v = (uint32_t)(uint8_t)vals[hh[q]];
                    v4 = (v4 & ~(0xFFu << (8 * q))) | v << (8 * q);
                }
            }
            if (all_rec && i + 3 < n_total) {
                *(uint32_t *)(s0 + i) = v4;
                *(uint32_t *)(s1 + i) = v4;
            } else {
                // only the slots with a record are written
                for (int q = 0; q < 4 && i + q < n_total; ++q) {
                    if (hh[q] < 0) continue;
                    const int8_t v = (int8_t)(v4 >> (8 * q));
                    s0[i + q] = v;
                    s1[i + q] = v;
                }
            }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (i + q < n_total && (int8_t)(v4 >> (8 * q)) == inf) nib |= 1u << q;
    }
    // lanes 16w .. 16w + 15 hold the 64 slots of word w of the wavefront's four
    uint64_t x = (uint64_t)nib << (4 * (lane & 15));
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) x |= (uint64_t)__shfl_xor((long long)x, off);
    if ((lane & 15) == 0 && i < n_total) bits[i >> 6] = x;
}

// Ghost refresh keyed by id: resolve through the map, then scatter.
__global__ void halo_unpack_ids_kernel(const unsigned long long *__restrict__ keys,
                                       const int32_t *__restrict__ mvals, int64_t cap,
                                       const int64_t *__restrict__ ids, const int8_t *__restrict__ vals,
                                       int64_t n, int8_t *s0, int8_t *s1, int32_t *misses) {
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= n) return;
    const int32_t s = map_find(keys, mvals, cap, ids[g]);
    if (s < 0) { atomicAdd(misses, 1); return; }
    s0[s] = vals[g];
    s1[s] = vals[g];
}

// Pack (gpu_kernels.py:852-909 gathers rows of the send list): out[h] = st[slots[h]].
// A slot outside [0, n_total) reads as 0 and sets *bad: the range check costs
// nothing here, where a pass over 72k slots on the host took 16 of a pack's 47 us.
__device__ __forceinline__ uint32_t state_at(const int8_t *__restrict__ st, int32_t slot, uint32_t n_total,
                                             uint32_t &wrong) {
    const bool in = (uint32_t)slot < n_total;
    wrong |= in ? 0u : 1u;
    return in ? (uint32_t)(uint8_t)st[slot] : 0u;
}

__global__ void gather_kernel(const int8_t *__restrict__ st, const int32_t *__restrict__ slots,
                              int8_t *__restrict__ out, int64_t n, uint32_t n_total, uint32_t *bad) {
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= n) return;
    uint32_t wrong = 0u;
    out[g] = (int8_t)state_at(st, slots[g], n_total, wrong);
    if (wrong && bad) *bad = 1u;
}

// The same as 2-bit codes, four records a byte (record h in bits 2 (h % 4)
// and 2 (h % 4) + 1 of byte h / 4); states are taken modulo 4.
__global__ void gather2_kernel(const int8_t *__restrict__ st, const int32_t *__restrict__ slots,
                               uint8_t *__restrict__ out, int64_t n, uint32_t n_total, uint32_t *bad) {
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (4 * j >= n) return;
    uint32_t b = 0u, wrong = 0u;
    if (4 * j + 4 <= n) {                               // one load of the four slots
        struct __attribute__((packed, aligned(4))) Four { int32_t s[4]; };
        const Four f = *(const Four *)(slots + 4 * j);
#pragma unroll
        for (int q = 0; q < 4; ++q) b |= (state_at(st, f.s[q], n_total, wrong) & 3u) << (2 * q);
    } else {
        for (int q = 0; 4 * j + q < n; ++q) b |= (state_at(st, slots[4 * j + q], n_total, wrong) & 3u) << (2 * q);
    }
    out[j] = (uint8_t)b;
    if (wrong && bad) *bad = 1u;
}

// 0x80 in every byte of x that equals the byte whose copies fill y.
__device__ __forceinline__ uint32_t eq_bytes(uint32_t x, uint32_t y) {
    const uint32_t t = x ^ y;
    return ~(((t & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | t) & 0x80808080u;
}

// Census of the local slots of one state buffer.  Block b writes its own row
// part[b][0..4]: agents in states 0..3, sum of the degrees of the agents in
// s_code.  A thread takes 16 agents at a time: one 16-byte load of states and
// one of the one-byte degrees (255: read the row bounds); both arrays are
// padded to whole groups of 64.  Bound by the loads' latency at small sizes
// and by the 2 bytes an agent at large ones.  The rows are summed on the host,
// straight from page-locked memory: adding them with atomics to five words,
// which run one after another, took 96 us a launch on 100k agents, this takes
// 4.1 us.
__global__ __launch_bounds__(256) void stats_kernel(const int8_t *__restrict__ st, const uint8_t *__restrict__ deg8,
                                                    const int64_t *__restrict__ row_ptr, int64_t n_local,
                                                    int8_t s_code, unsigned long long *__restrict__ part) {
    uint32_t cnt[4] = {0u, 0u, 0u, 0u};
    unsigned long long dsum = 0;
    const uint32_t S = 0x01010101u * (uint32_t)(uint8_t)s_code;
    for (int64_t i0 = 16 * ((int64_t)blockIdx.x * blockDim.x + threadIdx.x); i0 < n_local;
         i0 += 16 * (int64_t)gridDim.x * blockDim.x) {
        const uint4 x4 = *(const uint4 *)(st + i0), d4 = *(const uint4 *)(deg8 + i0);
        const uint32_t x[4] = {x4.x, x4.y, x4.z, x4.w}, d[4] = {d4.x, d4.y, d4.z, d4.w};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int64_t left = n_local - i0 - 4 * q;                     // agents from this word on
            const uint32_t in = left >= 4 ? ~0u : left <= 0 ? 0u : (1u << (8 * left)) - 1u;
#pragma unroll
            for (int s = 0; s < 4; ++s) cnt[s] += (uint32_t)__popc(eq_bytes(x[q], 0x01010101u * s) & in);
            const uint32_t sus = ((eq_bytes(x[q], S) & in) >> 7) * 0xFFu;
            dsum += __builtin_amdgcn_sad_u8(d[q] & sus, 0u, 0u);
            uint32_t big = eq_bytes(d[q], 0xFFFFFFFFu) & sus;              // rows of 255 entries or more
            while (big) {
                const int64_t i = i0 + 4 * q + (__ffs(big) - 1) / 8;
                big &= big - 1u;
                dsum += (unsigned long long)(row_ptr[i + 1] - row_ptr[i] - 255);
            }
        }
    }
    __shared__ unsigned long long red[256 / 64][5];
    unsigned long long v[5] = {cnt[0], cnt[1], cnt[2], cnt[3], dsum};
#pragma unroll
    for (int k = 0; k < 5; ++k) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) v[k] += __shfl_down(v[k], off);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][k] = v[k];
    }
    __syncthreads();
    if (threadIdx.x < 5) {
        unsigned long long t = 0;
        for (int w = 0; w < 256 / 64; ++w) t += red[w][threadIdx.x];
        part[SS_STATS_ROW * blockIdx.x + threadIdx.x] = t;
    }
}

// out[j] = st[slot[j]] for the n_local agents in the caller's order, ghost slots
// as they are.  A thread makes 16 bytes of the result: four 16-byte loads of
// slots (padded to whole groups of 16), 16 byte gathers, one 16-byte store.
// Bound by the gathers (one cache line each, the states stay in the last-level
// cache): 20 us for 10M agents into device memory, where scattering the
// downloaded states on the host took 13 ms; a readback has it write the chunks
// to page-locked memory, at the bus's rate.
__global__ __launch_bounds__(256) void order_kernel(const int8_t *__restrict__ st, const int32_t *__restrict__ slot,
                                                    int8_t *__restrict__ out, int64_t first, int64_t end,
                                                    int64_t n_local) {
    const int64_t j0 = first + 16 * ((int64_t)blockIdx.x * blockDim.x + threadIdx.x);
    if (j0 >= end) return;
    uint32_t w[4] = {0u, 0u, 0u, 0u};
    const bool whole = j0 + 16 <= n_local;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        int32_t x[4];
        if (whole) {
            const int4 v = *(const int4 *)(slot + j0 + 4 * q);
            x[0] = v.x; x[1] = v.y; x[2] = v.z; x[3] = v.w;
        } else {
#pragma unroll
            for (int h = 0; h < 4; ++h) {
                const int64_t j = j0 + 4 * q + h;
                x[h] = j < n_local ? slot[j] : j < end ? (int32_t)j : 0;
            }
        }
#pragma unroll
        for (int h = 0; h < 4; ++h) w[q] |= (uint32_t)(uint8_t)st[x[h]] << (8 * h);
    }
    *(uint4 *)(out + j0 - first) = make_uint4(w[0], w[1], w[2], w[3]);     // out is padded to whole groups of 16
}

// Page-locked host memory <-> device by the compute units, for what is waited
// for: bytes of src (W per lane, one byte per lane of the rest) and a table of
// words2 8-byte words.  Bound by the trip over the bus: 3.3 us for a halo and
// the descriptors, where the copy engine's hand-over to the compute stream and
// back costs some 25 us beside the 3 us of the copy, and the table took a copy
// of its own.
template <class W>
__global__ __launch_bounds__(256) void stage_kernel(const char *__restrict__ src, char *__restrict__ dst, int64_t bytes,
                                                    const uint64_t *__restrict__ src2, uint64_t *__restrict__ dst2,
                                                    int64_t words2) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t n = bytes / (int64_t)sizeof(W), rest = n * (int64_t)sizeof(W) + (i - n);
    if (i < n) ((W *)dst)[i] = ((const W *)src)[i];
    else if (rest < bytes) dst[rest] = src[rest];
    if (i < words2) dst2[i] = src2[i];
}

// Plain streaming copy (16 B per lane per step): the known-size reference for
// calibrating hardware traffic counters and the achievable HBM bandwidth.
__global__ void copy_kernel(const uint4 *__restrict__ src, uint4 *__restrict__ dst, int64_t n16) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += (int64_t)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

// n 4-byte reads at scattered positions of src (n_words words, far larger
// than the caches): the known-count random-gather reference for the traffic
// counters.  One word per thread is written so the reads stay.
__global__ void gather_probe_kernel(const uint32_t *__restrict__ src, int64_t n_words, int64_t n,
                                    uint32_t *__restrict__ out) {
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t acc = 0u;
    for (int64_t i = g; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const uint64_t h = (uint64_t)i * 0x9E3779B97F4A7C15ull;
        acc += src[(int64_t)((h >> 17) % (uint64_t)n_words)];
    }
    out[g] = acc;
}

__global__ void fill_u32_kernel(uint32_t *p, int64_t n, uint32_t v) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = v ^ (uint32_t)i;
}

// Range check of an uploaded CSR index array: first_bad = smallest e with
// col[e] outside [0, n_total) (stays ~0 when every entry is in range).
__global__ void check_cols_kernel(const int32_t *__restrict__ col, int64_t nnz, int64_t n_total,
                                  unsigned long long *first_bad) {
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < nnz; e += (int64_t)gridDim.x * blockDim.x) {
        const int32_t c = col[e];
        if (c < 0 || (int64_t)c >= n_total) atomicMin(first_bad, (unsigned long long)e);
    }
}

inline unsigned grid_for(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

}  // namespace

// ---- launchers (host) ----
hipError_t ss_launch_entries(const int64_t *row_ptr, const int32_t *col_idx, int64_t n_rows, int64_t nnz,
                             int64_t n_total, unsigned long long *part, int max_blocks, int *blocks, hipStream_t s) {
    *blocks = 0;
    if (nnz <= 0 || n_rows <= 0) return hipSuccess;
    *blocks = (int)std::min<int64_t>(max_blocks, (int64_t)grid_for(nnz, 16 * 256));
    hipLaunchKernelGGL(entries_kernel, dim3(*blocks), dim3(256), 0, s, row_ptr, col_idx, n_rows, nnz, n_total, part);
    return hipGetLastError();
}

hipError_t ss_launch_agents(int64_t *row_ptr, const int64_t *ids, int64_t n, int64_t n_total, int64_t nnz,
                            uint8_t *deg8, uint32_t *lo, int64_t *edge64, unsigned long long *part, int max_blocks,
                            int *blocks, hipStream_t s) {
    *blocks = (int)std::min<int64_t>(max_blocks, (int64_t)grid_for(n_total + 1, 256));
    hipLaunchKernelGGL(agents_kernel, dim3(*blocks), dim3(256), 0, s, row_ptr, ids, n, n_total, nnz, deg8, lo, edge64,
                       part);
    return hipGetLastError();
}

hipError_t ss_launch_high_words(const int64_t *ids, int64_t n, uint32_t *hi, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(high_words_kernel, dim3(grid_for(n, 256)), dim3(256), 0, s, ids, n, hi);
    return hipGetLastError();
}

hipError_t ss_launch_bits(const int8_t *st, uint64_t *bits, int64_t w0, int64_t w1, int64_t n_total, int8_t inf,
                          hipStream_t s) {
    if (w1 <= w0) return hipSuccess;
    hipLaunchKernelGGL(bits_kernel, dim3(grid_for((w1 - w0) * 64, 256)), dim3(256), 0, s, st, bits, w0, w1, n_total,
                       inf);
    return hipGetLastError();
}

hipError_t ss_launch_map_lookup(const unsigned long long *keys, const int32_t *vals, int64_t cap, const int64_t *ids,
                                int32_t *out, int64_t n, uint32_t *counts, bool lowest, int num_cus, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    const unsigned grid = std::min(grid_for(n, 256), (unsigned)num_cus * 8u);
    if (lowest)
        hipLaunchKernelGGL(map_lookup_kernel<true>, dim3(grid), dim3(256), 0, s, keys, vals, cap, ids, out, n, counts);
    else
        hipLaunchKernelGGL(map_lookup_kernel<false>, dim3(grid), dim3(256), 0, s, keys, vals, cap, ids, out, n, counts);
    return hipGetLastError();
}

hipError_t ss_launch_halo_records(const int32_t *slot, int64_t n, int64_t base, int32_t *rec, int64_t n_rec,
                                  hipStream_t s) {
    hipError_t e = ss_launch_fill_i32(rec, n_rec, -1, s);
    if (e != hipSuccess || n <= 0) return e;
    hipLaunchKernelGGL(halo_records_kernel, dim3(grid_for(n, 256)), dim3(256), 0, s, slot, n, base, rec);
    return hipGetLastError();
}

hipError_t ss_launch_halo_gather(int8_t *s0, int8_t *s1, const int8_t *cur, uint64_t *bits, const int32_t *rec,
                                 const int8_t *vals, int64_t base, int64_t n_total, int8_t inf, bool packed,
                                 hipStream_t s) {
    if (n_total <= base) return hipSuccess;
    if (packed)
        hipLaunchKernelGGL(halo_gather_kernel<true>, dim3(grid_for(n_total - base, 4 * 256)), dim3(256), 0, s, s0,
                           s1, cur, bits, rec, vals, base, n_total, inf);
    else
        hipLaunchKernelGGL(halo_gather_kernel<false>, dim3(grid_for(n_total - base, 4 * 256)), dim3(256), 0, s, s0,
                           s1, cur, bits, rec, vals, base, n_total, inf);
    return hipGetLastError();
}

hipError_t ss_launch_halo_unpack_ids(const unsigned long long *keys, const int32_t *mvals, int64_t cap,
                                     const int64_t *ids, const int8_t *vals, int64_t n, int8_t *s0, int8_t *s1,
                                     int32_t *misses, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(halo_unpack_ids_kernel, dim3(grid_for(n, 256)), dim3(256), 0, s, keys, mvals, cap, ids, vals,
                       n, s0, s1, misses);
    return hipGetLastError();
}

hipError_t ss_launch_gather(const int8_t *st, const int32_t *slots, int8_t *out, int64_t n, int64_t n_total,
                            uint32_t *bad, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(gather_kernel, dim3(grid_for(n, 256)), dim3(256), 0, s, st, slots, out, n, (uint32_t)n_total,
                       bad);
    return hipGetLastError();
}

hipError_t ss_launch_gather2(const int8_t *st, const int32_t *slots, uint8_t *out, int64_t n, int64_t n_total,
                             uint32_t *bad, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(gather2_kernel, dim3(grid_for((n + 3) / 4, 256)), dim3(256), 0, s, st, slots, out, n,
                       (uint32_t)n_total, bad);
    return hipGetLastError();
}

hipError_t ss_launch_fill_i32(int32_t *p, int64_t n, int32_t v, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(fill_i32_kernel, dim3(grid_for(n, 256)), dim3(256), 0, s, p, n, v);
    return hipGetLastError();
}

hipError_t ss_launch_stats(const int8_t *st, const uint8_t *deg8, const int64_t *row_ptr, int64_t n_local,
                           int8_t s_code, unsigned long long *part, int max_blocks, int *blocks, hipStream_t s) {
    *blocks = 0;
    if (n_local <= 0) return hipSuccess;
    *blocks = (int)std::min<int64_t>(max_blocks, (int64_t)grid_for(n_local, 16 * 256));
    hipLaunchKernelGGL(stats_kernel, dim3(*blocks), dim3(256), 0, s, st, deg8, row_ptr, n_local, s_code, part);
    return hipGetLastError();
}

hipError_t ss_launch_order(const int8_t *st, const int32_t *slot, int8_t *out, int64_t first, int64_t end,
                           int64_t n_local, hipStream_t s) {
    if (end <= first) return hipSuccess;
    hipLaunchKernelGGL(order_kernel, dim3(grid_for(end - first, 16 * 256)), dim3(256), 0, s, st, slot, out, first, end,
                       n_local);
    return hipGetLastError();
}

hipError_t ss_launch_stage(const void *src, void *dst, int64_t bytes, const uint64_t *src2, uint64_t *dst2,
                           int64_t words2, hipStream_t s) {
    // as wide as the pointers allow
    const uintptr_t at = (uintptr_t)src | (uintptr_t)dst;
    const int64_t w = at % 16 == 0 ? 16 : at % 4 == 0 ? 4 : 1;
    const int64_t lanes = std::max(bytes / w + bytes % w, words2);
    if (lanes <= 0) return hipSuccess;
    auto kernel = w == 16 ? stage_kernel<uint4> : w == 4 ? stage_kernel<uint32_t> : stage_kernel<uint8_t>;
    hipLaunchKernelGGL(kernel, dim3(grid_for(lanes, 256)), dim3(256), 0, s, (const char *)src, (char *)dst, bytes, src2,
                       dst2, words2);
    return hipGetLastError();
}

hipError_t ss_launch_copy(const void *src, void *dst, int64_t bytes, int grid, hipStream_t s) {
    hipLaunchKernelGGL(copy_kernel, dim3(grid), dim3(256), 0, s, (const uint4 *)src, (uint4 *)dst, bytes / 16);
    return hipGetLastError();
}

hipError_t ss_launch_gather_probe(const uint32_t *src, int64_t n_words, int64_t n, uint32_t *out, int grid,
                                  hipStream_t s) {
    hipLaunchKernelGGL(gather_probe_kernel, dim3(grid), dim3(256), 0, s, src, n_words, n, out);
    return hipGetLastError();
}

hipError_t ss_launch_fill_u32(uint32_t *p, int64_t n, uint32_t v, int grid, hipStream_t s) {
    hipLaunchKernelGGL(fill_u32_kernel, dim3(grid), dim3(256), 0, s, p, n, v);
    return hipGetLastError();
}

hipError_t ss_launch_check_cols(const int32_t *col, int64_t nnz, int64_t n_total, unsigned long long *first_bad,
                                int grid, hipStream_t s) {
    if (nnz <= 0) return hipSuccess;
    hipLaunchKernelGGL(check_cols_kernel, dim3(grid), dim3(256), 0, s, col, nnz, n_total, first_bad);
    return hipGetLastError();
}
