/*
 * gepi_stage.h -- panel staging kernels (replace the host transpose and
 * uploads of src/kernels/setup1.h:72-102 and the constant-memory class masks
 * of kernel1.cu:329-337).
 *
 * k_decode_bed     SNP-major .bed bytes -> [n_var][3][W64] planes on device
 *                  (BinPlinkReader.h:171-201: code 0 -> allele 1 + valid,
 *                  2 -> both + valid, 3 -> allele 2 + valid, 1 -> missing).
 * k_gather_class   per scan: samples reordered class-contiguously
 *                  (class 0 then class 1, each padded to 128 bits) into the
 *                  popcount layout [n_var_pad][3][wc] dwords.
 * k_transpose_k    popcount layout -> MFMA layout [n_ks][n_var_pad][3] of
 *                  64-sample words, so that one K step of a tile is contiguous.
 * k_qa_variants    missing calls per variant (one wave per variant)
 * k_qa_samples     missing calls per sample (a workgroup per 4,096 samples and
 *                  448 variants; partial counts added atomically)
 * k_gather_variants  copies the planes of selected variants to a new panel
 * k_class_f4       panel -> fp4 MFMA layout directly: per plane row, the
 *                  samples of each class are compressed (stable) out of the
 *                  file order with mask-driven bit compression, cut into
 *                  128-sample K steps and written four K steps at a time as
 *                  64-byte super-step rows (class 0, then class 1 from the
 *                  next super-step), with each row's set bits in the fourth
 *                  K steps; or three K steps at a time in the grouped
 *                  layout of the wave-tile count kernel.
 * The QA kernels replace the loops of checkQuality (src/reader/
 * PlinkReader.h:237-335), which count missing calls on the host.
 */
#ifndef GEPI_STAGE_H
#define GEPI_STAGE_H

#include "gepi_device.h"

namespace gepi {

/* The even bits of x as its low half. */
__device__ __forceinline__ uint32_t even_bits(uint64_t x) {
    x &= 0x5555555555555555ull;
    x = (x | (x >> 1)) & 0x3333333333333333ull;
    x = (x | (x >> 2)) & 0x0F0F0F0F0F0F0F0Full;
    x = (x | (x >> 4)) & 0x00FF00FF00FF00FFull;
    x = (x | (x >> 8)) & 0x0000FFFF0000FFFFull;
    return (uint32_t)(x | (x >> 16));
}

/* A thread per 64 samples of a variant: 16 bytes from anywhere in the payload,
 * as five aligned dwords (the buffer has BED_PAD bytes past the payload; what
 * lies past the row is masked), the two bits of the codes apart and from them
 * the planes.  Bound by the planes' writes: 50,000 x 4,000 106 -> 25 us against
 * one byte and one sample at a time.                                       */
constexpr int64_t BED_PAD = 32;
static __global__ void __launch_bounds__(256) k_decode_bed(const uint8_t *__restrict__ bed,
                                                           int64_t n_var, int32_t n_samples,
                                                           int32_t w64, int64_t bps,
                                                           uint64_t *__restrict__ nat,
                                                           uint32_t *__restrict__ any_missing) {
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= n_var * w64) return;
    const int64_t v = gid / w64;
    const int32_t wd = (int32_t)(gid - v * w64);
    const int64_t at = v * bps + 16 * (int64_t)wd;
    const uint32_t *src = reinterpret_cast<const uint32_t *>(bed + (at & ~3ll));
    const uint32_t sh = 8u * (uint32_t)(at & 3);
    uint32_t d[5];
#pragma unroll
    for (int i = 0; i < 5; i++) d[i] = src[i];
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; i++) w[i] = __builtin_amdgcn_alignbit(d[i + 1], d[i], sh);
    const uint64_t x0 = (uint64_t)w[1] << 32 | w[0], x1 = (uint64_t)w[3] << 32 | w[2];
    const uint64_t lo = (uint64_t)even_bits(x1) << 32 | even_bits(x0);
    const uint64_t hi = (uint64_t)even_bits(x1 >> 1) << 32 | even_bits(x0 >> 1);
    const int32_t left = n_samples - 64 * wd;
    const uint64_t in = left >= 64 ? ~0ull : (1ull << left) - 1ull;
    uint64_t *dst = nat + (v * 3) * w64 + wd;
    dst[0] = ~lo & in;              /* codes 0, 2 */
    dst[w64] = hi & in;             /* codes 2, 3 */
    const uint64_t valid = (~lo | hi) & in; /* all but 1  */
    dst[2 * w64] = valid;
    /* read first: one line of L2, written by few */
    if (valid != in &&
        __hip_atomic_load(any_missing, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0u)
        __hip_atomic_store(any_missing, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

/* out[v][p][d] bit b = panel bit perm[32*d + b] (0 for perm < 0 or v >= n_var). */
static __global__ void __launch_bounds__(256) k_gather_class(const uint64_t *__restrict__ nat,
                                                       int32_t n_var, int32_t w64,
                                                       const int32_t *__restrict__ perm,
                                                       int32_t wc, int32_t wused,
                                                       uint32_t *__restrict__ out) {
    extern __shared__ uint64_t srow[];
    const int32_t v = blockIdx.x;
    const bool real = v < n_var;
    for (int32_t i = threadIdx.x; i < 3 * w64; i += blockDim.x)
        srow[i] = real ? nat[(int64_t)v * 3 * w64 + i] : 0ull;
    __syncthreads();
    for (int32_t i = threadIdx.x; i < 3 * wc; i += blockDim.x) {
        int32_t p = i / wc, d = i - p * wc;
        uint32_t word = 0;
        if (real && d < wused) {
            const int32_t *pp = perm + 32 * d;
            const uint64_t *row = srow + p * w64;
#pragma unroll 8
            for (int32_t b = 0; b < 32; b++) {
                int32_t s = pp[b];
                if (s >= 0) word |= (uint32_t)((row[s >> 6] >> (s & 63)) & 1ull) << b;
            }
        }
        out[((int64_t)v * 3 + p) * wc + d] = word;
    }
}

/* Tile of 32 variants x 32 K steps per workgroup. */
static __global__ void __launch_bounds__(256) k_transpose_k(const uint32_t *__restrict__ cls,
                                                      int32_t n_var_pad, int32_t wc, int32_t n_ks,
                                                      uint64_t *__restrict__ out) {
    __shared__ uint64_t tile[96][33];
    const int32_t v0 = blockIdx.x * 32, s0 = blockIdx.y * 32;
    for (int32_t idx = threadIdx.x; idx < 96 * 32; idx += blockDim.x) {
        const int32_t vp = idx >> 5, k = idx & 31;
        const int32_t s = s0 + k;
        const int32_t v = v0 + vp / 3, p = vp % 3;
        uint64_t val = 0;
        if (s < n_ks)
            val = *reinterpret_cast<const uint64_t *>(cls + ((int64_t)v * 3 + p) * wc + 2 * s);
        tile[vp][k] = val;
    }
    __syncthreads();
    for (int32_t idx = threadIdx.x; idx < 96 * 32; idx += blockDim.x) {
        const int32_t k = idx / 96, vp = idx - 96 * k;
        const int32_t s = s0 + k;
        if (s < n_ks) out[((int64_t)s * n_var_pad + v0) * 3 + vp] = tile[vp][k];
    }
}

/* Compression of one 32-bit sample word for one class: x & m moved to the
 * low popc(m) bits, order kept, by five conditional shifts whose move masks
 * depend on m only (Hacker's Delight, "compress").  Built on the host once
 * per scan; the same for every plane row.                                   */
struct CompressWord {
    uint32_t m;     /* class mask word                                      */
    uint32_t mv[5]; /* move masks of the stages shifting by 1, 2, 4, 8, 16 */
    uint32_t cnt;   /* popc(m)                                              */
    uint32_t pad;
};

__host__ __device__ inline CompressWord make_compress_word(uint32_t m) {
    CompressWord c;
    c.m = m;
    c.cnt = 0;
    for (uint32_t t = m; t; t &= t - 1) c.cnt++;
    uint32_t mk = ~m << 1; /* zeros to the right of each position */
    for (int i = 0; i < 5; i++) {
        uint32_t mp = mk ^ (mk << 1); /* parallel suffix (xor) */
        mp ^= mp << 2;
        mp ^= mp << 4;
        mp ^= mp << 8;
        mp ^= mp << 16;
        const uint32_t mv = mp & m;
        c.mv[i] = mv;
        m = (m ^ mv) | (mv >> (1u << i));
        mk &= ~mp;
    }
    c.pad = 0;
    return c;
}

__device__ __forceinline__ uint32_t compress_word(uint32_t x, const CompressWord &c) {
    x &= c.m;
#pragma unroll
    for (int i = 0; i < 5; i++) {
        const uint32_t t = x & c.mv[i];
        x = (x ^ t) | (t >> (1u << i));
    }
    return x;
}

/* Bit n of the low byte of x moved to bit 4n (three shift-or-mask rounds). */
__device__ __forceinline__ uint32_t spread8(uint32_t x) {
    x &= 0xFFu;
    x = (x | (x << 12)) & 0x000F000Fu;
    x = (x | (x << 6)) & 0x03030303u;
    x = (x | (x << 3)) & 0x11111111u;
    return x;
}

/* One 64-byte super-step row of the fp4 layout from the row's four
 * 128-sample K steps k0..k3 (32-bit word g of a K step holds its samples
 * 32g .. 32g+31): dword d of 16-byte group g holds, at bit 4n + p, sample
 * 32g + 8d + n of K step p (bit 3, the e2m1 sign bit, for K step 3).      */
__device__ __forceinline__ uint4 super_group(uint32_t a, uint32_t b, uint32_t c, uint32_t e) {
    uint4 o;
    o.x = spread8(a) | (spread8(b) << 1) | (spread8(c) << 2) | (spread8(e) << 3);
    o.y = spread8(a >> 8) | (spread8(b >> 8) << 1) | (spread8(c >> 8) << 2) | (spread8(e >> 8) << 3);
    o.z = spread8(a >> 16) | (spread8(b >> 16) << 1) | (spread8(c >> 16) << 2) |
          (spread8(e >> 16) << 3);
    o.w = spread8(a >> 24) | (spread8(b >> 24) << 1) | (spread8(c >> 24) << 2) |
          (spread8(e >> 24) << 3);
    return o;
}

/* A stream of bits appended in order, cut into 128-sample K steps, and
 * written S (3 or 4) K steps at a time as super-step rows
 * out[(u * rows + r) * 4 + g]; with S = 4, pc3 counts the set bits of every
 * fourth K step (the count kernel's correction of that step).  GRP: the
 * grouped layout of the wave-tile kernel instead, uint4 g of row r = 3v + p
 * at out[(((u * NG + v / 32) * 3 + p) * 4 + g) * 32 + v % 32] (NG = rows /
 * 96 groups of 32 variants), so that the 32 variants of a group, one plane
 * and one 16-byte column, are 512 contiguous bytes.  Every thread
 * of a launch appends the same counts in the same order, so the bookkeeping
 * is uniform.  The completed K steps of the current super-step advance
 * through k0, k1, k2 (an indexed array would be placed in scratch memory). */
template <int S, bool GRP = false>
struct SuperStream {
    uint64_t acc;
    int32_t na, nq, np, pc3;
    int64_t u;
    uint32_t q0, q1, q2, q3;
    uint4 k0, k1, k2;

    __device__ __forceinline__ void init(int64_t u0) {
        acc = 0;
        na = nq = np = pc3 = 0;
        u = u0;
        q0 = q1 = q2 = q3 = 0;
        k0 = k1 = k2 = make_uint4(0u, 0u, 0u, 0u);
    }
    __device__ __forceinline__ void kstep(const uint4 &kr, uint4 *out, int64_t rows, int64_t r) {
        if (np == 0) {
            k0 = kr;
        } else if (np == 1) {
            k1 = kr;
        } else if (S == 4 && np == 2) {
            k2 = kr;
        } else {
            /* S = 3: kr is the third K step, bit 3 of every nibble stays 0 */
            const uint4 c = S == 4 ? k2 : kr, e = S == 4 ? kr : make_uint4(0u, 0u, 0u, 0u);
            if (r < rows) {
                /* GRP: uint4 g of the row is 32 uint4 after uint4 g - 1 */
                int64_t at, gs;
                if (GRP) {
                    const int64_t v = r / 3, pl = r - 3 * v;
                    at = (((u * (rows / 96) + (v >> 5)) * 3 + pl) * 4) * 32 + (v & 31);
                    gs = 32;
                } else {
                    at = (u * rows + r) * 4;
                    gs = 1;
                }
                uint4 *dst = out + at;
                dst[0] = super_group(k0.x, k1.x, c.x, e.x);
                dst[gs] = super_group(k0.y, k1.y, c.y, e.y);
                dst[2 * gs] = super_group(k0.z, k1.z, c.z, e.z);
                dst[3 * gs] = super_group(k0.w, k1.w, c.w, e.w);
            }
            pc3 += __popc(e.x) + __popc(e.y) + __popc(e.z) + __popc(e.w);
            u++;
        }
        np = np == S - 1 ? 0 : np + 1;
    }
    __device__ __forceinline__ void emit(uint32_t w, uint4 *out, int64_t rows, int64_t r) {
        q0 = q1;
        q1 = q2;
        q2 = q3;
        q3 = w;
        if (++nq == 4) {
            kstep(make_uint4(q0, q1, q2, q3), out, rows, r);
            nq = 0;
        }
    }
    __device__ __forceinline__ void append(uint32_t bits, int32_t k, uint4 *out, int64_t rows,
                                           int64_t r) {
        acc |= (uint64_t)bits << na;
        na += k;
        if (na >= 32) {
            emit((uint32_t)acc, out, rows, r);
            acc >>= 32;
            na -= 32;
        }
    }
    /* zero-pads the last K step and the last super-step of the stream */
    __device__ __forceinline__ void finish(uint4 *out, int64_t rows, int64_t r) {
        if (na > 0) {
            emit((uint32_t)acc, out, rows, r);
            acc = 0;
            na = 0;
        }
        while (nq != 0) emit(0u, out, rows, r);
        while (np != 0) kstep(make_uint4(0u, 0u, 0u, 0u), out, rows, r);
    }
};

/* One thread per plane row r = v*3 + p of [0, rows) (rows = n_var_pad * 3;
 * rows of padding variants v >= n_var are zero).  cw: [2][2*w64]
 * CompressWord, class 0 then class 1.  S K steps per super-step (4: single
 * scans, 3: the batch engine).  Class 0 fills super-steps [0, u1) (u1 =
 * f4_super or f4_super3 of its K steps), class 1 the super-steps from u1
 * on.  S = 4: pc3[c * rows + r] = set bits of row r in the fourth K steps
 * of class c's super-steps.  GRP: the grouped layout (SuperStream; rows a
 * multiple of 96).  The panel rows of a workgroup are staged
 * through LDS 8 words at a time (coalesced reads).                         */
constexpr int CLS_CHUNK = 8;
template <int S, bool GRP = false>
__global__ void __launch_bounds__(256) k_class_f4(const uint64_t *__restrict__ nat, int32_t n_var,
                                                   int32_t w64, const CompressWord *__restrict__ cw,
                                                   int64_t rows, int32_t u1,
                                                   uint4 *__restrict__ out,
                                                   int32_t *__restrict__ pc3) {
    __shared__ uint64_t srow[256][CLS_CHUNK + 1];
    const int64_t r0 = (int64_t)blockIdx.x * 256;
    const int64_t r = r0 + threadIdx.x;
    const int64_t real_rows = (int64_t)n_var * 3;
    SuperStream<S, GRP> s0, s1;
    s0.init(0);
    s1.init(u1);
    const CompressWord *c0 = cw, *c1 = cw + 2 * w64;
    for (int32_t base = 0; base < w64; base += CLS_CHUNK) {
        __syncthreads();
        for (int32_t idx = threadIdx.x; idx < 256 * CLS_CHUNK; idx += 256) {
            const int32_t rl = idx / CLS_CHUNK, wd = idx % CLS_CHUNK;
            const int64_t rr = r0 + rl;
            uint64_t val = 0;
            if (rr < real_rows && base + wd < w64) val = nat[rr * w64 + base + wd];
            srow[rl][wd] = val;
        }
        __syncthreads();
        const int32_t nw = w64 - base < CLS_CHUNK ? w64 - base : CLS_CHUNK;
        for (int32_t wd = 0; wd < nw; wd++) {
            const uint64_t x = srow[threadIdx.x][wd];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const uint32_t xh = (uint32_t)(x >> (32 * h));
                const int32_t j = 2 * (base + wd) + h;
                const CompressWord a = c0[j], b = c1[j];
                if (a.cnt) s0.append(compress_word(xh, a), (int32_t)a.cnt, out, rows, r);
                if (b.cnt) s1.append(compress_word(xh, b), (int32_t)b.cnt, out, rows, r);
            }
        }
    }
    s0.finish(out, rows, r);
    s1.finish(out, rows, r);
    if (S == 4 && r < rows) {
        pc3[r] = s0.pc3;
        pc3[rows + r] = s1.pc3;
    }
}

/* Where a super-step's 384 class samples lie in the panel's file order: from
 * bit `skip` of the class's samples in 32-bit word j0, up to word j1. */
struct SuperSrc {
    int32_t cls, j0, skip, j1;
};

/* Class layout of the wave tiles on genotype planes (count_f4g_unit): the
 * grouped layout with plane 0 = homozygous for allele 1 (a1 & ~a2), 1 =
 * heterozygous (a1 & a2), 2 = homozygous for allele 2.  blockIdx.x: 64
 * variants, a wave per plane; blockIdx.y: the super-step, whose samples the
 * host has located (src), so that a scan's super-steps are made in parallel
 * (one thread for a row's whole sample range took 384 us for 8,000 x 20,001
 * and 38 us for 20,000 x 2,048).  blockIdx.y = n_u: the variants' shares of
 * missing calls among the class samples, rounded up, or, with margin > 0, the
 * margins that the products of a panel without missing calls leave out
 * (F4GMargins), `margin` added to the totals.                              */
constexpr int CLSG_THREADS = 192;
static __global__ void __launch_bounds__(CLSG_THREADS)
    k_class_geno(const uint64_t *__restrict__ nat, int32_t n_var, int32_t w64,
                 const CompressWord *__restrict__ cw, const SuperSrc *__restrict__ src, int32_t n_u,
                 int32_t n0, int32_t n, float margin, uint4 *__restrict__ out,
                 float *__restrict__ miss) {
    __shared__ uint64_t row[2][64][CLS_CHUNK + 1];
    __shared__ int32_t sum[4][64];
    const int tid = threadIdx.x, p = tid >> 6, vl = tid & 63;
    const int32_t v0 = blockIdx.x * 64, u = blockIdx.y;
    auto stage = [&](int32_t w0) {
        /* words w0 .. w0 + 7 of the allele planes of the 64 variants */
        __syncthreads();
        for (int i = tid; i < 2 * 64 * CLS_CHUNK; i += CLSG_THREADS) {
            const int wd = i % CLS_CHUNK, v = (i / CLS_CHUNK) & 63, pl = i / (64 * CLS_CHUNK);
            const bool in = v0 + v < n_var && w0 + wd < w64;
            row[pl][v][wd] = in ? nat[((int64_t)(v0 + v) * 3 + pl) * w64 + w0 + wd] : 0ull;
        }
        __syncthreads();
    };
    if (u == n_u) {
        for (int i = tid; i < 256; i += CLSG_THREADS) sum[i >> 6][i & 63] = 0;
        /* margin = 0: valid calls; else homozygous 1 and heterozygous, by class */
        int32_t k[4] = {0, 0, 0, 0};
        for (int32_t w0 = 0; w0 < w64; w0 += CLS_CHUNK) {
            stage(w0);
            const int32_t nw = w64 - w0 < CLS_CHUNK ? w64 - w0 : CLS_CHUNK;
            for (int32_t wd = p; wd < nw; wd += 3) { /* the waves share the words */
                const uint64_t a1 = row[0][vl][wd], a2 = row[1][vl][wd];
                const CompressWord *a = cw + 2 * (w0 + wd), *b = a + 2 * w64;
                const uint64_t m0 = ((uint64_t)a[1].m << 32) | a[0].m;
                const uint64_t m1 = ((uint64_t)b[1].m << 32) | b[0].m;
                const uint64_t x = margin == 0.0f ? a1 | a2 : a1 & ~a2, y = margin == 0.0f ? 0ull : a1 & a2;
                k[0] += __popcll(x & m0);
                k[1] += __popcll(x & m1);
                k[2] += __popcll(y & m0);
                k[3] += __popcll(y & m1);
            }
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 4; i++) atomicAdd(&sum[i][vl], k[i]);
        __syncthreads();
        if (p != 0) return;
        const int32_t x0 = sum[0][vl], x1 = sum[1][vl], y0 = sum[2][vl], y1 = sum[3][vl];
        if (margin == 0.0f) {
            miss[v0 + vl] = n > 0 ? (float)(n - x0 - x1) / (float)n * (1.0f + 1e-6f) : 0.0f;
        } else {
            float *o = miss + (int64_t)(v0 + vl) * 6;
            o[0] = (float)(x0 + x1) + margin;
            o[1] = (float)(y0 + y1) + margin;
            o[2] = (float)(n - x0 - x1 - y0 - y1) + margin;
            o[3] = (float)x0;
            o[4] = (float)y0;
            o[5] = (float)(n0 - x0 - y0);
        }
        return;
    }
    const SuperSrc s = src[u];
    const CompressWord *c = cw + (int64_t)s.cls * 2 * w64;
    uint64_t acc = 0;
    int32_t na = 0, nq = 0, skip = s.skip;
    uint32_t q[12]; /* the last 12 words made; the oldest first */
#pragma unroll
    for (int i = 0; i < 12; i++) q[i] = 0;
    auto emit = [&](uint32_t w) {
#pragma unroll
        for (int i = 0; i < 11; i++) q[i] = q[i + 1];
        q[11] = w;
        nq++;
    };
    for (int32_t w0 = s.j0 >> 1; 2 * w0 < s.j1; w0 += CLS_CHUNK) {
        stage(w0);
        for (int32_t wd = 0; wd < CLS_CHUNK; wd++) {
            const uint64_t a1 = row[0][vl][wd], a2 = row[1][vl][wd];
            const uint64_t x = p == 0 ? a1 & ~a2 : p == 1 ? a1 & a2 : a2 & ~a1;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int32_t j = 2 * (w0 + wd) + h;
                if (j < s.j0 || j >= s.j1) continue;
                const CompressWord m = c[j];
                acc |= (uint64_t)(compress_word((uint32_t)(x >> (32 * h)), m) >> skip) << na;
                na += (int32_t)m.cnt - skip;
                skip = 0;
                if (na >= 32 && nq < 12) {
                    emit((uint32_t)acc);
                    acc >>= 32;
                    na -= 32;
                }
            }
        }
    }
    /* a class's last super-step: zero-padded */
    if (nq < 12) emit((uint32_t)acc);
    while (nq < 12) emit(0u);
    const int64_t G = blockIdx.x * 2 + (vl >> 5), NG = (int64_t)gridDim.x * 2;
    uint4 *dst = out + (((int64_t)u * NG + G) * 3 + p) * 128 + (vl & 31);
#pragma unroll
    for (int g = 0; g < 4; g++) dst[32 * g] = super_group(q[g], q[4 + g], q[8 + g], 0u);
}

/* missing[v] = n_samples - popc(valid plane of variant v); 64 threads per
 * variant.  Samples beyond n_samples are never valid in a panel. */
static __global__ void __launch_bounds__(256) k_qa_variants(const uint64_t *__restrict__ nat,
                                                            int64_t n_var, int32_t w64,
                                                            int32_t n_samples,
                                                            int32_t *__restrict__ missing) {
    const int64_t v = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (v >= n_var) return;
    const uint64_t *valid = nat + (v * 3 + 2) * w64;
    int32_t c = 0;
    for (int32_t w = lane; w < w64; w += 64) c += __popcll(valid[w]);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off);
    if (lane == 0) missing[v] = n_samples - c;
}

/* valid[s] += number of variants with a call for sample s; grid (variants /
 * QA_VARS, words / 64).  missing = n_var - valid is taken on the host.  A lane
 * holds a 64-sample word column, a wave a quarter of the block's variants;
 * seven words are added at a time into three bit planes of counters (carry-save
 * adders, about two operations a word), which are spread over the word's 64
 * counters in LDS when they are full.  50,000 x 4,000: 281 -> 18 us against a
 * thread per sample, which read every word 64 times.                       */
constexpr int QA_VARS = 448;
static __global__ void __launch_bounds__(256) k_qa_samples(const uint64_t *__restrict__ nat,
                                                           int64_t n_var, int32_t w64,
                                                           int32_t n_samples,
                                                           int32_t *__restrict__ valid_count) {
    __shared__ uint32_t cnt[64][65]; /* [bit][word], padded */
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int i = threadIdx.x; i < 64 * 64; i += 256) cnt[i >> 6][i & 63] = 0u;
    __syncthreads();
    const int32_t w = blockIdx.y * 64 + lane;
    const int64_t v0 = (int64_t)blockIdx.x * QA_VARS + wave * (QA_VARS / 4);
    const int64_t v1 = v0 + QA_VARS / 4 < n_var ? v0 + QA_VARS / 4 : n_var;
    if (w < w64) {
        const uint64_t *col = nat + 2 * (int64_t)w64 + w;
        const int64_t stride = 3 * (int64_t)w64;
        uint64_t p[7] = {0, 0, 0, 0, 0, 0, 0}; /* bit planes of the counters */
        for (int64_t v = v0; v < v1; v += 7) {
            uint64_t x[7];
#pragma unroll
            for (int i = 0; i < 7; i++) x[i] = v + i < v1 ? col[(v + i) * stride] : 0ull;
            auto sum = [](uint64_t a, uint64_t b, uint64_t c) { return a ^ b ^ c; };
            auto maj = [](uint64_t a, uint64_t b, uint64_t c) { return (a & b) | (c & (a | b)); };
            const uint64_t s0 = sum(x[0], x[1], x[2]), c0 = maj(x[0], x[1], x[2]);
            const uint64_t s1 = sum(x[3], x[4], x[5]), c1 = maj(x[3], x[4], x[5]);
            uint64_t add[3];
            add[0] = sum(s0, s1, x[6]);
            const uint64_t c2 = maj(s0, s1, x[6]);
            add[1] = sum(c0, c1, c2);
            add[2] = maj(c0, c1, c2);
            uint64_t carry = 0; /* p += add: at most QA_VARS / 4 = 112 < 128 */
#pragma unroll
            for (int i = 0; i < 7; i++) {
                const uint64_t b = i < 3 ? add[i] : 0ull, t = p[i] ^ b;
                const uint64_t o = t ^ carry;
                carry = (p[i] & b) | (t & carry);
                p[i] = o;
            }
        }
#pragma unroll 4
        for (int b = 0; b < 64; b++) {
            uint32_t c = 0;
#pragma unroll
            for (int i = 0; i < 7; i++) c |= (uint32_t)((p[i] >> b) & 1ull) << i;
            atomicAdd(&cnt[b][lane], c);
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 64 * 64; i += 256) {
        const int32_t s = blockIdx.y * 4096 + i;
        const uint32_t c = cnt[i & 63][i >> 6];
        if (s < n_samples && c) atomicAdd(&valid_count[s], (int32_t)c);
    }
}

/* dst variant i = src variant idx[i]: its three plane rows of w64 words. */
static __global__ void __launch_bounds__(256) k_gather_variants(const uint64_t *__restrict__ src,
                                                                const int64_t *__restrict__ idx,
                                                                int64_t n_keep, int32_t w64,
                                                                uint64_t *__restrict__ dst) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t per = (int64_t)3 * w64;
    if (t >= n_keep * per) return;
    const int64_t i = t / per, o = t - i * per;
    dst[i * per + o] = src[idx[i] * per + o];
}

} // namespace gepi

#endif
