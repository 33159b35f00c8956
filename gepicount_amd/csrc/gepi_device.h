/*
 * gepi_device.h -- device-side records, scan state and the fused per-pair
 * filter shared by the count kernels.
 */
#ifndef GEPI_DEVICE_H
#define GEPI_DEVICE_H

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "../../include/gepicount.h"
#include "gepi_score.h"

namespace gepi {

constexpr int TV = 32;              /* popcount kernel: variants per tile side       */
constexpr int TM = 64;              /* MFMA kernel: variants per tile side           */
constexpr int SEL_SMALL = 1024;     /* radix select finishes in LDS below this size  */
constexpr int MFMA_LOW_MAX = 16383; /* class count limit of the 0x01-encoded class   */
constexpr int64_t TILE_EVALS_MAX = (int64_t)TM * TM * 20; /* evaluations of the largest tile */

/* A candidate for the top-k: exact score plus counts.  32 bytes. */
struct Cand {
    double score;
    uint64_t idx; /* sA << 32 | sB << 3 | fun */
    uint32_t w, x, y, z;
};

/* A record read or written field by field: as a copy of the struct half of an
 * array of them stays in private memory, and the runtime allocates device
 * memory for a queue's first kernel with any (24 MiB here).               */
__device__ __forceinline__ Cand load_cand(const Cand *p) {
    return Cand{p->score, p->idx, p->w, p->x, p->y, p->z};
}
__device__ __forceinline__ void store_cand(Cand *p, const Cand &c) {
    p->score = c.score;
    p->idx = c.idx;
    p->w = c.w;
    p->x = c.x;
    p->y = c.y;
    p->z = c.z;
}

/* An evaluation that passed the single-precision filter.  16 bytes. */
struct Pend {
    uint16_t w, x, y, z;
    uint64_t idx;
};

/* The threshold fields have a 256-byte line pair of their own: no launch
 * that reads them writes them, while every workgroup's reservations hit the
 * counters after them (see filter_consts).                                */
struct ScanState {
    double thr_score;          /* admission key: (thr_score, thr_idx), inclusive   */
    uint64_t thr_idx;
    float filt_k;              /* entropy filter coefficient, 0 = admit everything */
    float filt_t;              /* entropy: the threshold in nats, rounded down     */
    uint32_t thr_pad[58];
    uint32_t full;             /* the band's pending list overflowed (band_full): a
                                * line of its own, written by few               */
    uint32_t full_pad[63];
    uint32_t overflow;         /* candidate buffer overflowed in this band          */
    uint32_t pad2;
    unsigned long long count;  /* records in the active candidate buffer           */
    unsigned long long count2; /* records written by a compaction                  */
    unsigned long long pend_count;
    uint32_t pend_overflow;
    uint32_t pad1;
    unsigned long long pair_count; /* variant pairs put off in this band (k_pairs)  */
    /* radix select */
    uint64_t key_hi, key_lo;
    uint32_t bits_done, rank, matched, done, gather_n, pad0;
    uint32_t hist[256];
};

static_assert(offsetof(ScanState, full) == 256 && offsetof(ScanState, overflow) == 512,
              "thresholds and the overflow mark share no line with counters");

struct CountArgs {
    const uint32_t *planes;   /* popcount layout [n_var_pad][3][wc] dwords          */
    const uint64_t *planes_k; /* int8: [n_ks][n_var_pad][3] 64-sample words;
                               * fp4: [n_u][n_var_pad*3][4] uint4 super-step rows
                               * (K steps of 128 samples: 4 per super-step for
                               * single scans, 3 in the batch engine; see
                               * k_class_f4)                                      */
    const int32_t *pc3;       /* fp4 single scans: [2][n_var_pad*3] set bits of
                               * each plane row in its class's fourth K steps
                               * (k_class_f4); unused by the batch engine         */
    int64_t tile_begin;       /* first linear tile of the band                      */
    int32_t n_tiles;          /* tiles in the band (= grid size)                    */
    int32_t n_var;
    int32_t n_var_pad;
    int32_t wc;               /* dwords per plane row (multiple of 32)              */
    int32_t w0;               /* class-0 dwords (multiple of 4)                     */
    int32_t wused;            /* dwords holding data (multiple of 4)                */
    int32_t n_ks;             /* K steps: 64 samples (int8), 128 samples (fp4)      */
    int32_t ks0;              /* K steps of class 0 (fp4: class 1 starts at
                               * super-step f4_super(ks0))                         */
    int32_t cls0_high;        /* MFMA: class 0 encoded as 0x80 (else class 1 is)    */
    int32_t f32;              /* fp4: class sizes for which the filter may work on
                               * the fp32 counts (f32_counts)                    */
    int32_t n0, n1;           /* class sizes (bounds of y and z: Fisher filter)   */
    /* wave tiles on genotype planes (count_f4g_unit): per variant the share
     * of missing calls [n_var_pad], or the margins [n_var_pad][6] of a panel
     * without missing calls (F4GMargins); p = n0/n, k, 2 p (1-p), 2 p (1-p) n; the
     * accumulators' start and what it takes off the screen's right side    */
    const float *miss;
    float sc_p, sc_k, sc_q, sc_m, sc_start, sc_sub;
    float h0, h1;             /* chi-square coefficient per nat: h0 + h1 min(y, z)
                               * (chi2_slope)                                     */
    uint4 *pairs;             /* pairs that passed the screen, for k_pairs: 3 (without
                               * missing calls 2) uint4 each; null with pair_cap 0                       */
    uint32_t pair_cap;
    int32_t watch;            /* workgroups look whether the band is full (band_full) */
    int32_t pair_from;        /* units before this one test their pairs in the kernel
                               * (pairs_from)                                     */
    ScanState *st;
    Pend *pend;
    unsigned long long pcap;
    const double *lfact;      /* ln t! (Fisher filter)                              */
    struct PairRec *park;     /* fp4 wave tiles, Fisher: [park_slots][park_cap]
                               * regions for parked variant pairs (null: none)   */
    uint32_t *park_busy;      /* [park_slots] claim flags, then 8 claim counters  */
    uint32_t park_cap, park_slots;
};

/* The XCD (0-7) this wave runs on, from the hardware register. */
__device__ __forceinline__ uint32_t xcc_id() {
    return (uint32_t)__builtin_amdgcn_s_getreg((3 << 11) | (0 << 6) | 20) & 7u; /* HW_REG_XCC_ID */
}

/* A parking region of CountArgs::park for this workgroup (thread 0): the
 * first free slot, from a rotating start, among the slots of the XCD it
 * runs on.  The XCDs' L2 caches are not coherent with one another, so a
 * region written and read through one XCD's L2 must not pass through
 * another's within a launch (a region reused across XCDs read stale
 * records when another XCD's dirty lines were written back over it).
 * Every claim is released before its workgroup ends and the host keeps
 * more slots per XCD than workgroups can be resident on one, so a free
 * slot is found; the probes are bounded all the same (PARK_NONE: no
 * region, the pairs are finished in the lane).                           */
constexpr uint32_t PARK_NONE = 0xFFFFFFFFu;
__device__ __forceinline__ uint32_t park_claim(uint32_t *busy, uint32_t slots) {
    const uint32_t x = xcc_id(), per = slots >> 3, base = x * per;
    uint32_t s = atomicAdd(&busy[slots + x], 1u) % per;
    for (uint32_t t = 0; t < 4 * per; t++) {
        if (atomicCAS(&busy[base + s], 0u, 1u) == 0u) return base + s;
        s = s + 1 == per ? 0u : s + 1;
    }
    return PARK_NONE;
}

__host__ __device__ inline void tile_of(int64_t t, int32_t &ta, int32_t &tb) {
    /* t = ta*(ta+1)/2 + tb, 0 <= tb <= ta */
    double r = sqrt(8.0 * (double)t + 1.0);
    int64_t a = (int64_t)((r - 1.0) * 0.5);
    while (a * (a + 1) / 2 > t) a--;
    while ((a + 1) * (a + 2) / 2 <= t) a++;
    ta = (int32_t)a;
    tb = (int32_t)(t - a * (a + 1) / 2);
}

/* Workgroup tile t of a scan with n_a A blocks: A variants [64ta, 64ta+64)
 * against B variants [32tb, 32tb+32), 0 <= tb <= 2ta+1 (row ta holds 2ta+2
 * tiles, so n_a(n_a+1) in all).  Tiles are numbered in panels of
 * F4_PANEL rows; panel rows [a0, a0+P) take indices [a0(a0+1),
 * (a0+P)(a0+P+1)), first the rectangle tb < 2a0+2 that all of them share,
 * column by column, then the rest of each row (row a0+i has 2i more tiles)
 * in row order.  Workgroups running together on one XCD take consecutive
 * tiles, so they share 8 A blocks and 8 B blocks in that XCD's L2; in row
 * order they shared one A block and read 64 B blocks that the next row
 * needs again only after the whole row has gone through.                 */
constexpr int F4_PANEL = 8;
__host__ __device__ inline void tile_of_f4(int64_t t, int32_t n_a, int32_t &ta, int32_t &tb) {
    double r = sqrt(4.0 * (double)t + 1.0);
    int64_t a = (int64_t)((r - 1.0) * 0.5);
    while (a * (a + 1) > t) a--;
    while ((a + 1) * (a + 2) <= t) a++;
    const int64_t a0 = a - a % F4_PANEL;
    const int64_t P = n_a - a0 < F4_PANEL ? n_a - a0 : F4_PANEL;
    const int64_t W = 2 * a0 + 2;
    const int64_t l = t - a0 * (a0 + 1);
    int64_t ra, rb;
    if (l < P * W) {
        rb = P == F4_PANEL ? l / F4_PANEL : l / P; /* a shift for a full panel */
        ra = a0 + (l - rb * P);
    } else {
        const int64_t e = l - P * W; /* i(i-1) tiles of the rest precede row a0+i */
        int64_t i = 1;
        while ((i + 1) * i <= e) i++;
        ra = a0 + i;
        rb = W + e - i * (i - 1);
    }
    ta = (int32_t)ra;
    tb = (int32_t)rb;
}

/* Linear workgroup tile of variant pair (a >= b).  Square tiles of side tv
 * (popcount, int8 MFMA): ta*(ta+1)/2 + tb.  fp4 tiles of 64 x 32 variants
 * (n_a4 > 0, the scan's A blocks): the inverse of tile_of_f4 at ta = a/64,
 * tb = b/32.                                                              */
__host__ __device__ inline int64_t tile_index(int64_t a, int64_t b, int32_t tv, int32_t n_a4) {
    if (n_a4 > 0) {
        const int64_t ta = a / 64, tb = b / 32;
        const int64_t a0 = ta - ta % F4_PANEL;
        const int64_t P = n_a4 - a0 < F4_PANEL ? n_a4 - a0 : F4_PANEL;
        const int64_t W = 2 * a0 + 2, i = ta - a0;
        return a0 * (a0 + 1) + (tb < W ? tb * P + i : P * W + i * (i - 1) + (tb - W));
    }
    const int64_t ta = a / tv, tb = b / tv;
    return ta * (ta + 1) / 2 + tb;
}

/* Workgroup -> tile of the band.  Consecutive workgroups are dispatched to
 * the 8 XCDs round robin; each XCD gets a contiguous run of tiles, so that
 * the tiles running together on it are neighbours in the tile order and
 * share panel rows in that XCD's L2.                                      */
__device__ __forceinline__ int64_t band_tile(int64_t tile_begin, int32_t n_tiles) {
    const int32_t gidx = blockIdx.x;
    const int32_t xcd = gidx & 7, slot = gidx >> 3;
    const int32_t per = n_tiles >> 3, rem = n_tiles & 7;
    return tile_begin + (int64_t)xcd * per + (xcd < rem ? xcd : rem) + slot;
}

/* Survivors of one workgroup are staged in LDS (LDS atomics) and written to
 * the pending list with one global reservation per workgroup; past
 * PEND_LDS they go to the pending list directly.                          */
constexpr int PEND_LDS = 256;
template <int N>
struct PendStageN {
    static constexpr uint32_t cap = N;
    Pend rec[N];
    uint32_t n;
    uint32_t full; /* the pending list was found full: no more is tested */
    unsigned long long base;
};
typedef PendStageN<PEND_LDS> PendStage;

/* Atomics on the scan state through global-address-space pointers: the
 * state pointer may come from a descriptor in memory, where the compiler
 * cannot tell its address space, and global atomics on a uniform address
 * let it combine a wave's atomics into one (generic ones it does not). */
typedef __attribute__((address_space(1))) unsigned long long gu64_t;
typedef __attribute__((address_space(1))) uint32_t gu32_t;
__device__ __forceinline__ unsigned long long st_add(unsigned long long *p, unsigned long long v) {
    return __hip_atomic_fetch_add((gu64_t *)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_or(uint32_t *p, uint32_t v) {
    __hip_atomic_fetch_or((gu32_t *)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

/* A pending list that is full: its band is redone whatever else it finds, so
 * workgroups and loops that have not begun leave their work out where g.watch
 * asks them to look (the band of a guessed threshold, which may pass nearly
 * every evaluation; looking costs 20,000 x 2,048 0.8% of its time, and 1.9%
 * in every band).                                                         */
__device__ __forceinline__ void mark_full(const CountArgs &g) {
    st_or(&g.st->pend_overflow, 1u);
    __hip_atomic_store((gu32_t *)&g.st->full, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ bool band_full(const CountArgs &g) {
    return g.watch && __hip_atomic_load((gu32_t *)&g.st->full, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u;
}

/* Places for n records of every active lane (n < 32): `at` in the stage for
 * the first `own` of them, `gat` in the pending list for the others.  One LDS
 * atomic per wave, and one global one where the stage is full: under a loose
 * threshold most records go there, and one per record of a lane kept the
 * count kernel waiting (top-1,000,000 of 20,000 x 2,048: first band 6.3 ms,
 * all 23.2; now 0.76 and 7.4).                                             */
struct PushSlots {
    uint32_t at, own;
    unsigned long long gat;
};
template <class PS>
__device__ __forceinline__ PushSlots push_reserve(const CountArgs &g, PS &ps, uint32_t n) {
    uint32_t before = 0, total = 0;
#pragma unroll
    for (int b = 0; b < 5; b++) {
        const uint64_t m = __ballot((n >> b) & 1u);
        before += __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                            __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u)) << b;
        total += (uint32_t)__popcll(m) << b;
    }
    const uint64_t act = __ballot(true);
    const bool lead = (int)__lane_id() == __builtin_ctzll(act);
    uint32_t base = 0;
    if (lead) base = atomicAdd(&ps.n, total);
    base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
    PushSlots s;
    s.at = base + before;
    s.own = s.at < PS::cap ? (PS::cap - s.at < n ? PS::cap - s.at : n) : 0u;
    s.gat = 0;
    if (base + total > PS::cap) {
        const uint32_t room = base < PS::cap ? PS::cap - base : 0u, rest = total - room;
        uint32_t lo = 0, hi = 0;
        if (lead) {
            const unsigned long long q = st_add(&g.st->pend_count, (unsigned long long)rest);
            lo = (uint32_t)q;
            hi = (uint32_t)(q >> 32);
            if (q + rest > g.pcap) {
                mark_full(g);
                ps.full = 1;
            }
        }
        lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)lo);
        hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)hi);
        s.gat = ((unsigned long long)hi << 32 | lo) + (before > room ? before - room : 0u);
    }
    return s;
}

/* The next record of a lane into its places. */
template <class PS>
__device__ __forceinline__ void push_pending(const CountArgs &g, PS &ps, PushSlots &s, int32_t w,
                                             int32_t x, int32_t y, int32_t z, uint64_t idx) {
    Pend p;
    p.w = (uint16_t)w;
    p.x = (uint16_t)x;
    p.y = (uint16_t)y;
    p.z = (uint16_t)z;
    p.idx = idx;
    if (s.own) {
        ps.rec[s.at++] = p;
        s.own--;
    } else {
        if (s.gat < g.pcap) g.pend[s.gat] = p;
        s.gat++;
    }
}

/* Called by every thread of the workgroup at kernel start (before the first
 * barrier) and after the last push, respectively.                          */
template <class PS>
__device__ __forceinline__ void stage_init(PS &ps) {
    if (threadIdx.x == 0) {
        ps.n = 0;
        ps.full = 0;
    }
}
template <class PS>
__device__ __forceinline__ bool stage_full(PS &ps) {
    return __hip_atomic_load(&ps.full, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) != 0u;
}

/* The flush proper: every push is complete (the caller has passed a
 * barrier after the last push).                                           */
template <class PS>
__device__ __forceinline__ void stage_flush_after_barrier(const CountArgs &g, PS &ps) {
    if (threadIdx.x == 0) {
        const uint32_t n = ps.n < PS::cap ? ps.n : PS::cap;
        ps.n = n;
        ps.base = n ? st_add(&g.st->pend_count, (unsigned long long)n) : 0ull;
        if (n && ps.base + n > g.pcap) mark_full(g);
    }
    __syncthreads();
    const uint32_t n = ps.n;
    for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) {
        const unsigned long long pos = ps.base + i;
        if (pos < g.pcap) g.pend[pos] = ps.rec[i];
    }
}

template <class PS>
__device__ __forceinline__ void stage_flush(const CountArgs &g, PS &ps) {
    __syncthreads();
    stage_flush_after_barrier(g, ps);
}

/* Per-scan filter constants, read once per workgroup (filter_consts). */
struct FilterConsts {
    double thr_s; /* admission score threshold                                 */
    float kf;     /* entropy: chi-square coefficient, 0 = admit everything      */
    float kt;     /* entropy: threshold in nats                                */
    float k0, k1; /* entropy: another, k0 + k1 min(y, z); the larger one counts */
    float h0, h1; /* Fisher: the same per nat                                   */
    float a_s;    /* Fisher: -(thr + 1e-6) ln 10 - ln(2.55 n) / 2, less a
                   * float error margin                                        */
};

/* The thresholds through the constant address space: scalar loads from the
 * scalar cache.  As plain loads they became vector loads wherever an atomic
 * or a scheduling barrier precedes them, and shared a line with the pending
 * counter that every workgroup updates, so each workgroup waited for that
 * line before its filter (20,000 x 2,048, 2^15 workgroups: 3.24 ms against
 * 1.85 ms).                                                                */
__device__ __forceinline__ FilterConsts filter_consts(const ScanState *st, const CountArgs &g) {
    const auto *c = (const __attribute__((address_space(4))) ScanState *)(uintptr_t)st;
    FilterConsts fc;
    fc.thr_s = c->thr_score;
    fc.kf = c->filt_k;
    fc.h0 = g.h0;
    fc.h1 = g.h1;
    fc.kt = c->filt_t;
    fc.k0 = c->filt_t * g.h0;
    fc.k1 = c->filt_t * g.h1;
    const int32_t n0 = g.n0, n1 = g.n1;
    const double a = -(fc.thr_s + 1e-6) * 2.302585092994046;
    const double A = a - 0.5 * log(2.55 * (double)(n0 + n1 > 1 ? n0 + n1 : 1));
    /* the float roundings of A and of the per-pair arithmetic stay far
     * under this margin, which keeps the derived bound conservative        */
    fc.a_s = fc.thr_s < 0.0 ? (float)(A - (fabs(A) + fabs(a) + 10.0) * 1e-6) : 0.0f;
    return fc;
}

/* Counts of the four row pairs (2A+ia, 2B+ib) of a variant pair, rp = 2ia+ib,
 * for function f: with n = N11, a = NA, b = NB and v = V of one class,
 *   f = 0 AND n, 1 NAND b-n, 2 ANDN a-n, 3 NANDN v-a-b+n, 4 XOR a+b-2n.      */
__device__ __forceinline__ int32_t fun_count(int f, int32_t n, int32_t a, int32_t b, int32_t v) {
    return f == 0 ? n : f == 1 ? b - n : f == 2 ? a - n : f == 3 ? v - a - b + n : a + b - 2 * n;
}

/* Fisher's exact check of one evaluation: log10 P(obs) <= thr (p >=
 * P(observed table)) from the log-factorial table, with the admission's
 * 1e-6 margin.                                                             */
__device__ __forceinline__ bool fisher_admits(const CountArgs &g, const FilterConsts &fc, int32_t w,
                                              int32_t x, int32_t y, int32_t z) {
    const int32_t m = y + z;
    const double *lf = g.lfact;
    const double lp = ((lf[y] + lf[z]) + (lf[w + x] + lf[m - w - x])) -
                      (((lf[w] + lf[y - w]) + (lf[x] + lf[z - x])) + lf[m]);
    return lp * 0.4342944819032518 - 1e-6 <= fc.thr_s;
}

/* t log2 t in float. */
__device__ __forceinline__ float tlog2(int32_t t) {
    return t > 0 ? (float)t * __builtin_amdgcn_logf((float)t) : 0.0f;
}

/* Entropy's near-exact check of one evaluation: -I m (bits) <= thr m in float
 * sums of t log2 t.  The nine terms and their sum are within 6.2e-6 m log2 m
 * of the exact value (log2 and products to 2^-22 relative, eight additions
 * of at most 4 m log2 m to 2^-24), so the margin of 8e-6 keeps every
 * evaluation that the exact score admits.  c = L(y) + L(z) - L(m).  The
 * chi-square bound alone admits two to six times as many, each a pending
 * record and an exact score (top-1,000,000 of 20,000 x 2,048: 33.0M survivors
 * in 52 ms of count launches, 16.2M in 26 with this check).                */
__device__ __forceinline__ bool entropy_admits(float lim, float c, int32_t w, int32_t x, int32_t y,
                                               int32_t z) {
    const float s = c + (tlog2(w + x) + tlog2(y + z - w - x)) -
                    ((tlog2(w) + tlog2(y - w)) + (tlog2(x) + tlog2(z - x)));
    return s <= lim;
}

/* Appends the evaluations whose bit 5*rp+f is set in mask to the pending
 * list.  Runs only for lanes with a survivor.  The row pair's operands
 * advance through rotating registers: selecting among the counts with a
 * runtime index would place them in scratch memory.  The survivors of the
 * chi-square bound are checked first: entropy's by entropy_admits, Fisher's
 * against log10 P(obs) <= thr (p >= P(observed table)) with the
 * log-factorial table; a second walk over those left writes the records into
 * places reserved for the wave.                                            */
template <int FFUN, class PS>
__device__ __forceinline__ void push_mask(const CountArgs &g, PS &ps, const FilterConsts &fc,
                                          int32_t A, int32_t B, const int32_t (&c)[2][3][3],
                                          uint32_t mask) {
    if (stage_full(ps)) return; /* the band is redone */
    const int32_t y = c[0][2][2], z = c[1][2][2];
    /* body(bit, w, x) for the evaluations in mb4, row pair by row pair */
    auto walk = [&](uint32_t mb4, auto body) {
        int32_t n0a = c[0][0][0], n0b = c[0][0][1], n0c = c[0][1][0], n0d = c[0][1][1];
        int32_t n1a = c[1][0][0], n1b = c[1][0][1], n1c = c[1][1][0], n1d = c[1][1][1];
        int32_t a0 = c[0][0][2], a1 = c[1][0][2];
        int32_t b0 = c[0][2][0], b1 = c[1][2][0], b0o = c[0][2][1], b1o = c[1][2][1];
#pragma unroll 1
        for (int rp = 0; rp < 4; rp++) {
            uint32_t mb = (mb4 >> (5 * rp)) & 31u;
            while (mb) {
                const int f = __builtin_ctz(mb);
                mb &= mb - 1;
                body(rp, f, fun_count(f, n0a, a0, b0, y), fun_count(f, n1a, a1, b1, z));
            }
            n0a = n0b; n0b = n0c; n0c = n0d;
            n1a = n1b; n1b = n1c; n1c = n1d;
            if (rp == 1) { a0 = c[0][1][2]; a1 = c[1][1][2]; }
            int32_t t = b0; b0 = b0o; b0o = t;
            t = b1; b1 = b1o; b1o = t;
        }
    };
    uint32_t ok = mask; /* those that pass it */
    if (FFUN == GEPI_FFUNC_ENTROPY) {
        const float lm = tlog2(y + z), mf = (float)(y + z);
        const float lc = tlog2(y) + tlog2(z) - lm;
        const float ts = (float)fc.thr_s; /* +infinity before the first threshold */
        const float lim = ts < 0.0f ? ts * mf * (1.0f - 1e-6f) + 8e-6f * lm + 1e-6f : __builtin_inff();
        ok = 0;
        walk(mask, [&](int rp, int f, int32_t w, int32_t x) {
            ok |= entropy_admits(lim, lc, w, x, y, z) ? 1u << (5 * rp + f) : 0u;
        });
    } else if (fc.thr_s < 0.0) {
        ok = 0;
        walk(mask, [&](int rp, int f, int32_t w, int32_t x) {
            ok |= fisher_admits(g, fc, w, x, y, z) ? 1u << (5 * rp + f) : 0u;
        });
    }
    if (!ok) return;
    PushSlots s = push_reserve(g, ps, (uint32_t)__popc(ok));
    walk(ok, [&](int rp, int f, int32_t w, int32_t x) {
        push_pending(g, ps, s, w, x, y, z,
                     pack_idx(2 * (int64_t)A + (rp >> 1), 2 * (int64_t)B + (rp & 1), f));
    });
}

/* Filters the 20 (or 12 on the diagonal) evaluations of variant pair (A, B)
 * from the nine plane products of each class, c[cls][p][q] =
 * popc(planeA[p] & planeB[q] & class cls) with p, q in {allele1, allele2,
 * valid}.  Survivors are staged for the pending list.
 *
 * Both objectives reduce to a chi-square test.  With I the mutual
 * information of the class x f table (nats) and chi2/m = D^2/(y z q),
 * D = wz - xy, q = xx(m - xx), Jensen on the KL divergence gives
 * I <= ln(1 + chi2/m), so I >= T requires D^2 >= expm1(T) * y * z * q.
 * The second bound is I <= g(p) chi2/m with p = min(y, z)/m and g(p) =
 * -ln(1-p) (1-p)/p, the largest ratio of KL(a||p) to (a-p)^2/(p(1-p)) over
 * a (at the end a = 0; I is the mean of the KL terms of f = 0 and f = 1 and
 * chi2/m that of the quadratic ones): I >= T requires D^2 >= T/g(p) * y z q.
 * 1/g runs from 1 at p = 0 to 1.44 at 1/2 and is convex, so its tangent at
 * the scan's class fraction, taken at min(y, z)/(n0+n1) <= p, is a lower
 * bound (chi2_slope); the larger of the two coefficients is used.  Tables
 * near the threshold have small T, so with even classes a table needs
 * 1.44 times the chi-square to pass (entropy, top-1,000 of 20,000 x 2,048: 5.79 -> 3.69
 * ms, Fisher 7.47 -> 5.99; large scan 120.4 -> 116.6).
 * Entropy: -I_bits <= thr needs T = -thr * ln 2 (kf = 2^-thr - 1 and T made
 * where the threshold is updated, rounded down).
 * Fisher: p >= P(obs) = C(y,w) C(z,x) / C(m,xx).  For 1 <= k <= n-1
 *     sqrt(n / (8 k (n-k))) <= C(n,k) e^{-nH(k/n)} <= sqrt(n / (2 pi k (n-k)))
 * (H in nats), and C(n,0) = C(n,n) = 1 meets the left side as 1.  With X =
 * min(xx, m-xx) <= m/2 (a table and its complement have the same P and I):
 * w(y-w)/y <= w, x(z-x)/z <= x, w x <= X^2/4 and X(m-X)/m >= X/2, so
 * P(obs) >= e^{-mI} sqrt(2 pi (X/2) / (64 X^2/4)) = e^{-mI} / sqrt(5.1 X) >=
 * e^{-mI} / sqrt(2.55 m); with w or x at an end of its range P(obs) >=
 * e^{-mI} sqrt(pi/8), which is no less for m >= 1.  So log10 P(obs) - 1e-6 <=
 * thr needs
 *     T = (-(thr + 1e-6) ln 10 - ln(2.55 m) / 2) / m
 * (taken at ln(2.55 n) >= ln(2.55 m), one log per workgroup; bounding the
 * numerator and the denominator each by its own worst case cost ln(4yz)/2 -
 * 0.92, 2.4 nats more at 2,048 samples and 3 at 8,192);
 * its survivors are then checked exactly against the log-factorial table.
 * The test is s = fd^2 - RN(K*y*z*(1 - 2^-16) * q) > bias with fd = float(D)
 * squared exactly inside one fma.  fd is D exactly when |D| <= 2^24 (always
 * so on the float path) and within 2^-24 relative otherwise; the right side
 * is within 2^-21 relative; the 2^-16 shrink of K covers both, so every
 * table meeting the exact bound passes.  D == 0 (an independent table,
 * I == 0) fails whenever K > 0, and K == 0 (bias -1) admits everything.
 * D and xx are linear in the three per-row-pair quantities (N11, NA, NB):
 * up to sign, D_f = {Dn, Db-Dn, Da-Dn, (Da-Dn)+Db, (Da-Dn)+(Db-Dn)} with
 * Dq = q0*z - q1*y (only D^2 enters the test), and xx_f likewise from
 * S = q0 + q1.
 * A row pair is flagged when the largest of its five s exceeds the bias;
 * the bits of the functions are rebuilt, from the same expressions, only
 * for the lanes with a flagged row pair.
 *
 * ROLLED: a runtime loop over the four row pairs keeps the code of callers
 * with many pairs per thread small; its operands advance through rotating
 * registers (an indexed array would be placed in scratch memory).
 * DEFER: a variant pair with a flagged row pair is parked in pl (its counts)
 * for pair_drain instead of being finished in the lane.                    */
template <typename DT>
struct RowTest {
    float kyz, mf, bias;
    float kyzm; /* float counts: kyz * mf, exact (see filter_pair) */
    /* s of the five functions of one row pair.  Every D below is one
     * function's w z - x y up to sign, so |D| <= y z: exact for int32 and,
     * when y z <= 2^24, for float.                                         */
    __device__ __forceinline__ void s5(DT Dn, float Sn, DT Da, float Sa, DT Db, float Sb,
                                       float (&s)[5]) const {
        const DT Dnb = Db - Dn, Dna = Da - Dn;
        const DT D[5] = {Dn, Dnb, Dna, Dna + Db, Dna + Dnb};
        const float Sab = Sa + Sb;
        const float X[5] = {Sn, Sb - Sn, Sa - Sn, (mf - Sab) + Sn, Sab - 2.0f * Sn};
#pragma unroll
        for (int f = 0; f < 5; f++) {
            float r;
            if constexpr (sizeof(DT) == sizeof(float) && DT(0.5f) != DT(0)) {
                /* kyz (m - X) exactly in one fma, then one rounding */
                r = X[f] * __builtin_fmaf(-kyz, X[f], kyzm);
            } else {
                r = kyz * (X[f] * (mf - X[f]));
            }
            const float fd = (float)D[f];
            s[f] = __builtin_fmaf(fd, fd, -r);
        }
    }
    __device__ __forceinline__ bool any(DT Dn, float Sn, DT Da, float Sa, DT Db, float Sb) const {
        float s[5];
        s5(Dn, Sn, Da, Sa, Db, Sb, s);
        return fmaxf(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3])), s[4]) > bias;
    }
    __device__ __forceinline__ uint32_t bits(DT Dn, float Sn, DT Da, float Sa, DT Db, float Sb) const {
        float s[5];
        s5(Dn, Sn, Da, Sa, Db, Sb, s);
        uint32_t b = 0;
#pragma unroll
        for (int f = 0; f < 5; f++) b |= s[f] > bias ? (1u << f) : 0u;
        return b;
    }
};

/* Class sizes for which the fp4 filter works on its fp32 accumulators:
 * every product of a class-0 and a class-1 count exact in float (n0 n1 <=
 * 2^24) and m <= 16384 (the RowTest's exact kyz (m - X)).                  */
__host__ __device__ inline bool f32_counts(int64_t n0, int64_t n1) {
    return n0 * n1 <= ((int64_t)1 << 24) && n0 + n1 <= 16384;
}

/* Count arithmetic of the filter.  int32 counts (< 2^16): D = q0 z - q1 y
 * with 24-bit products.  float counts (the fp4 path's accumulators, exact
 * integers, f32_counts): every product q0 z, q1 y is at most n0 n1 <= 2^24
 * (a count of class c is at most n_c) and so exact, and fma gives D exactly
 * with no conversion.                                                     */
__device__ __forceinline__ int32_t dq_of(int32_t q0, int32_t q1, int32_t y, int32_t z) {
    return __mul24(q0, z) - __mul24(q1, y);
}
__device__ __forceinline__ float dq_of(float q0, float q1, float y, float z) {
    return __builtin_fmaf(q0, z, -(q1 * y));
}
__device__ __forceinline__ float sq_of(int32_t q0, int32_t q1) { return (float)(q0 + q1); }
__device__ __forceinline__ float sq_of(float q0, float q1) { return q0 + q1; }
__device__ __forceinline__ float yz_of(int32_t y, int32_t z) { return (float)__mul24(y, z); }
__device__ __forceinline__ float yz_of(float y, float z) { return y * z; }

struct PairList;
template <int FFUN, bool ROLLED, bool DEFER = false, typename CT, typename PL = PairList, class PS>
__device__ __forceinline__ void filter_pair(const CountArgs &g, PS &ps, const FilterConsts &fc,
                                            int32_t A, int32_t B, const CT (&c)[2][3][3],
                                            PL *pl = nullptr, const CT (*tot)[3] = nullptr,
                                            uint32_t rows_known = 0);

/* Variant pairs with a flagged row pair, parked in LDS: the lanes that
 * flag one are few and scattered over the waves, and finishing a pair (the
 * function bits, Fisher's exact check, the pending list) in the lane costs
 * each wave its full length for them.  After the tile the workgroup
 * finishes the parked pairs one per thread (pair_drain); past PAIR_LDS the
 * lane finishes at once.  Counts are below 2^16 (class sizes <= 46,340). */
constexpr int PAIR_LDS = 512;
struct PairRec {
    uint16_t c[2][3][3];
    int32_t A, B;
    uint32_t pad;
};
struct PairList {
    PairRec rec[PAIR_LDS];
    uint32_t n;
    uint32_t pad[3];
    __device__ __forceinline__ uint32_t cap() const { return PAIR_LDS; }
    __device__ __forceinline__ PairRec &at(uint32_t i) { return rec[i]; }
};

/* The same list with its records in global memory (a workgroup's own
 * region, L2-resident while the workgroup runs) and its counter in LDS. */
struct PairListG {
    uint32_t *n; /* LDS */
    PairRec *rec;
    uint32_t cap_;
    __device__ __forceinline__ uint32_t cap() const { return cap_; }
    __device__ __forceinline__ PairRec &at(uint32_t i) { return rec[i]; }
};
__device__ __forceinline__ uint32_t park_reserve(PairList *pl) { return atomicAdd(&pl->n, 1u); }
__device__ __forceinline__ uint32_t park_reserve(PairListG *pl) { return atomicAdd(pl->n, 1u); }

template <int FFUN, bool ROLLED, bool DEFER, typename CT, typename PL, class PS>
__device__ __forceinline__ void filter_pair(const CountArgs &g, PS &ps, const FilterConsts &fc,
                                            int32_t A, int32_t B, const CT (&c)[2][3][3],
                                            PL *pl, const CT (*tot)[3], uint32_t rows_known) {
    /* tot: the products' totals over both classes, c[0] + c[1], when the
     * caller holds them (the wave tiles' accumulators), else summed here */
    const CT y = c[0][2][2], z = c[1][2][2];
    const CT m = tot ? tot[2][2] : y + z;
    const float mf = (float)m;
    const float mn = (float)(y < z ? y : z);
    float K = fmaxf(fc.kf, __builtin_fmaf(fc.k1, mn, fc.k0));
    if (FFUN == GEPI_FFUNC_FISHERPV) {
        K = 0.0f;
        if (fc.thr_s < 0.0) {
            /* T = a_s / m, and K = T (1 + T/2) <= expm1(T) or T (h0 + h1
             * min(y, z)) <= T/g(p): both only lower K                      */
            const float r = __builtin_amdgcn_rcpf(m > 1 ? mf : 1.0f);
            const float T = fc.a_s * r;
            if (T > 0.0f)
                K = T * fmaxf(1.0f + 0.5f * T, __builtin_fmaf(fc.h1, mn, fc.h0)) * (1.0f - 2e-5f);
        }
    }
    RowTest<CT> rt;
    rt.kyz = K * yz_of(y, z) * (1.0f - 1.0f / 65536.0f);
    rt.mf = mf;
    rt.kyzm = 0.0f;
    if constexpr (sizeof(CT) == sizeof(float) && CT(0.5f) != CT(0)) {
        /* float counts come with m <= 16384 (14 bits): kyz cut down to 10
         * significant bits makes kyz m and kyz X exact, so that fma(-kyz, X,
         * kyz m) is kyz (m - X) exactly; cutting only lowers the bound */
        rt.kyz = __uint_as_float(__float_as_uint(rt.kyz) & 0xFFFFC000u);
        rt.kyzm = rt.kyz * mf;
    }
    rt.bias = K == 0.0f ? -1.0f : 0.0f;
    auto dq = [&](CT q0, CT q1) { return dq_of(q0, q1, y, z); };
    /* S of product (p, q): both classes' count */
    auto sq = [&](int p, int q) { return tot ? (float)tot[p][q] : sq_of(c[0][p][q], c[1][p][q]); };
    const CT Da0 = dq(c[0][0][2], c[1][0][2]), Da1 = dq(c[0][1][2], c[1][1][2]);
    const CT Db0 = dq(c[0][2][0], c[1][2][0]), Db1 = dq(c[0][2][1], c[1][2][1]);
    const float Sa0 = sq(0, 2), Sa1 = sq(1, 2);
    const float Sb0 = sq(2, 0), Sb1 = sq(2, 1);
    /* row pair rp = 2ia + ib flagged in bit rp; rows_known: flagged before
     * the pair was parked (that test is as conservative as this one) */
    uint32_t rows = 0;
    if (rows_known) {
        rows = rows_known;
    } else if (ROLLED) {
        CT n0a = c[0][0][0], n0b = c[0][0][1], n0c = c[0][1][0], n0d = c[0][1][1];
        CT n1a = c[1][0][0], n1b = c[1][0][1], n1c = c[1][1][0], n1d = c[1][1][1];
        CT Da = Da0, Db = Db0, Dbo = Db1;
        float Sa = Sa0, Sb = Sb0, Sbo = Sb1;
#pragma unroll 1
        for (int rp = 0; rp < 4; rp++) {
            rows |= rt.any(dq(n0a, n1a), sq_of(n0a, n1a), Da, Sa, Db, Sb) ? 1u << rp : 0u;
            n0a = n0b; n0b = n0c; n0c = n0d;
            n1a = n1b; n1b = n1c; n1c = n1d;
            if (rp == 1) { Da = Da1; Sa = Sa1; }
            CT t = Db; Db = Dbo; Dbo = t;
            float u = Sb; Sb = Sbo; Sbo = u;
        }
    } else {
        rows = (rt.any(dq(c[0][0][0], c[1][0][0]), sq(0, 0), Da0, Sa0, Db0, Sb0) ? 1u : 0u) |
               (rt.any(dq(c[0][0][1], c[1][0][1]), sq(0, 1), Da0, Sa0, Db1, Sb1) ? 2u : 0u) |
               (rt.any(dq(c[0][1][0], c[1][1][0]), sq(1, 0), Da1, Sa1, Db0, Sb0) ? 4u : 0u) |
               (rt.any(dq(c[0][1][1], c[1][1][1]), sq(1, 1), Da1, Sa1, Db1, Sb1) ? 8u : 0u);
    }
    if (A == B) rows &= ~2u; /* (2A, 2A+1) is not a row pair */
    if (DEFER && rows) {
        const uint32_t pos = park_reserve(pl);
        if (pos < pl->cap()) {
            PairRec &r = pl->at(pos);
#pragma unroll
            for (int k = 0; k < 2; k++)
#pragma unroll
                for (int p = 0; p < 3; p++)
#pragma unroll
                    for (int q = 0; q < 3; q++) r.c[k][p][q] = (uint16_t)c[k][p][q];
            r.A = A;
            r.B = B;
            r.pad = rows; /* the drain starts from these rows */
            return;
        }
    }
    if (rows) {
        /* rare: the function bits of the flagged row pairs */
        uint32_t mask = 0;
        if (rows & 1u)
            mask |= rt.bits(dq(c[0][0][0], c[1][0][0]), sq(0, 0), Da0, Sa0, Db0, Sb0);
        if (rows & 2u)
            mask |= rt.bits(dq(c[0][0][1], c[1][0][1]), sq(0, 1), Da0, Sa0, Db1, Sb1) << 5;
        if (rows & 4u)
            mask |= rt.bits(dq(c[0][1][0], c[1][1][0]), sq(1, 0), Da1, Sa1, Db0, Sb0) << 10;
        if (rows & 8u)
            mask |= rt.bits(dq(c[0][1][1], c[1][1][1]), sq(1, 1), Da1, Sa1, Db1, Sb1) << 15;
        int32_t ci[2][3][3];
#pragma unroll
        for (int k = 0; k < 2; k++)
#pragma unroll
            for (int p = 0; p < 3; p++)
#pragma unroll
                for (int q = 0; q < 3; q++) ci[k][p][q] = (int32_t)c[k][p][q];
        push_mask<FFUN>(g, ps, fc, A, B, ci, mask);
    }
}

/* Finishes the parked pairs, one per thread, with the int32 filter (as
 * conservative as the test that parked them, so it keeps every evaluation
 * that the exact top-k needs).  Every thread of the workgroup, after a
 * barrier that follows the last park; the caller clears pl.n after a later
 * barrier.                                                                 */
template <int FFUN>
__device__ __forceinline__ void pair_drain(const CountArgs &g, PendStage &ps, const FilterConsts &fc,
                                           const PairRec *rec, uint32_t n) {
    for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) {
        const PairRec &r = rec[i];
        int32_t c[2][3][3];
#pragma unroll
        for (int k = 0; k < 2; k++)
#pragma unroll
            for (int p = 0; p < 3; p++)
#pragma unroll
                for (int q = 0; q < 3; q++) c[k][p][q] = r.c[k][p][q];
        filter_pair<FFUN, true>(g, ps, fc, r.A, r.B, c, (PairList *)nullptr,
                                (const int32_t(*)[3]) nullptr, r.pad);
    }
}

/* Waits until every global store of this wave has been acknowledged by L2
 * (s_waitcnt vmcnt(0); expcnt and lgkmcnt at their maxima: no wait). */
__device__ __forceinline__ void f4_wait_stores() { __builtin_amdgcn_s_waitcnt(0x0F70); }

} // namespace gepi

#endif
