/*
 * gepi_sort.h -- the final ranking on the device: a scan's k candidate
 * records sorted by the canonical key and written as results.  Replaces the
 * host's sort of the whole list (the reference sorts on the device per tile
 * and on the host at the end, src/kernels/kernel1.cu:448,
 * src/kernels/misc1.cu:234-264).
 *
 * A merge sort: workgroups sort tiles of 2,048 records in LDS, then runs are
 * merged pairwise, every workgroup producing 2,048 records of the merged run
 * (its place in the two runs by a binary search along the merge path, the
 * records' ranks by binary searches in LDS).  Keys are distinct, so equal
 * elements need no rule.  Bound by memory traffic: each pass reads and writes
 * the list once (80 MB for 1,000,000 records: 72 us for the tiles, then 9
 * merges of 24; the host's sort took 82 ms).
 */
#ifndef GEPI_SORT_H
#define GEPI_SORT_H

#include "gepi_device.h"

namespace gepi {

constexpr int SORT_TILE = 2048;
constexpr int SORT_THREADS = 512;
constexpr int SORT_PER = SORT_TILE / SORT_THREADS;

struct SortKey {
    uint64_t hi, lo;
};
__device__ __forceinline__ SortKey key_of(const Cand &c) { return SortKey{order_bits(c.score), c.idx}; }
__device__ __forceinline__ bool key_lt(const SortKey &a, const SortKey &b) {
    return a.hi < b.hi || (a.hi == b.hi && a.lo < b.lo);
}

/* Tiles of SORT_TILE records of src, each sorted, to dst (not in place): a
 * bitonic sort of (key, place in the tile) in LDS; places past n sort last. */
static __global__ void __launch_bounds__(SORT_THREADS)
    k_sort_tiles(const Cand *__restrict__ src, Cand *__restrict__ dst, int64_t n) {
    __shared__ uint64_t hi[SORT_TILE], lo[SORT_TILE];
    __shared__ uint16_t at[SORT_TILE];
    const int64_t t0 = (int64_t)blockIdx.x * SORT_TILE;
    for (int i = threadIdx.x; i < SORT_TILE; i += SORT_THREADS) {
        SortKey k{~0ull, ~0ull};
        if (t0 + i < n) k = key_of(src[t0 + i]);
        hi[i] = k.hi;
        lo[i] = k.lo;
        at[i] = (uint16_t)i;
    }
    for (int size = 2; size <= SORT_TILE; size <<= 1) {
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            __syncthreads();
            for (int h = threadIdx.x; h < SORT_TILE / 2; h += SORT_THREADS) {
                const int i = 2 * h - (h & (stride - 1)), j = i + stride;
                const bool up = (i & size) == 0;
                const bool gt = hi[i] > hi[j] || (hi[i] == hi[j] && lo[i] > lo[j]);
                if (gt == up) {
                    const uint64_t a = hi[i], b = lo[i];
                    const uint16_t c = at[i];
                    hi[i] = hi[j];
                    lo[i] = lo[j];
                    at[i] = at[j];
                    hi[j] = a;
                    lo[j] = b;
                    at[j] = c;
                }
            }
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < SORT_TILE; i += SORT_THREADS)
        if (t0 + i < n) dst[t0 + i] = src[t0 + at[i]];
}

/* How many of the first `diag` records of the merge of a[0, na) and b[0, nb)
 * come from a. */
__device__ __forceinline__ int64_t merge_split(const Cand *a, int64_t na, const Cand *b, int64_t nb,
                                               int64_t diag) {
    int64_t lo = diag > nb ? diag - nb : 0, hi = diag < na ? diag : na;
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (key_lt(key_of(a[mid]), key_of(b[diag - 1 - mid])))
            lo = mid + 1;
        else
            hi = mid;
    }
    return lo;
}

/* Runs of `run` records (a multiple of SORT_TILE) of src merged pairwise. */
static __global__ void __launch_bounds__(SORT_THREADS)
    k_merge(const Cand *__restrict__ src, Cand *__restrict__ dst, int64_t n, int64_t run) {
    __shared__ uint64_t hi[SORT_TILE], lo[SORT_TILE];
    __shared__ int64_t split[2];
    const int64_t o0 = (int64_t)blockIdx.x * SORT_TILE, p0 = o0 / (2 * run) * (2 * run);
    const int64_t na = n - p0 < run ? n - p0 : run, nb0 = n - p0 - na, nb = nb0 < run ? nb0 : run;
    const Cand *a = src + p0, *b = a + na;
    const int64_t d0 = o0 - p0, dn = na + nb - d0 < SORT_TILE ? na + nb - d0 : SORT_TILE;
    if ((threadIdx.x & 63) == 0 && threadIdx.x < 128) {
        const int w = threadIdx.x >> 6;
        split[w] = merge_split(a, na, b, nb, d0 + (w ? dn : 0));
    }
    __syncthreads();
    const int64_t a0 = split[0], b0 = d0 - a0;
    const int ca = (int)(split[1] - a0), cb = (int)dn - ca;
    Cand c[SORT_PER];
#pragma unroll
    for (int u = 0; u < SORT_PER; u++) {
        const int i = threadIdx.x + u * SORT_THREADS;
        if (i < (int)dn) {
            c[u] = load_cand(i < ca ? a + a0 + i : b + b0 + i - ca);
            const SortKey k = key_of(c[u]);
            hi[i] = k.hi;
            lo[i] = k.lo;
        }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < SORT_PER; u++) {
        const int i = threadIdx.x + u * SORT_THREADS;
        if (i >= (int)dn) continue;
        /* own place in its run plus the smaller ones of the other */
        const SortKey k = key_of(c[u]);
        const int base = i < ca ? ca : 0;
        int l = 0, h = i < ca ? cb : ca;
        while (l < h) {
            const int mid = (l + h) >> 1;
            if (key_lt(SortKey{hi[base + mid], lo[base + mid]}, k))
                l = mid + 1;
            else
                h = mid;
        }
        store_cand(dst + o0 + (i < ca ? i : i - ca) + l, c[u]);
    }
}

/* Sorted records as results. */
static __global__ void __launch_bounds__(256)
    k_results(const Cand *__restrict__ src, gepi_result *__restrict__ dst, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const Cand c = src[i];
    gepi_result r;
    r.sA = (int64_t)(c.idx >> 32);
    r.sB = (int64_t)((c.idx >> 3) & 0x1FFFFFFFull);
    r.fun = (int32_t)(c.idx & 7);
    r.w = (int32_t)c.w;
    r.x = (int32_t)c.x;
    r.y = (int32_t)c.y;
    r.z = (int32_t)c.z;
    r.obj = c.score;
    r.reserved = 0;
    dst[i] = r;
}

} // namespace gepi

#endif
