/*
 * gepi_host.h -- host-side state shared by the library's HIP translation
 * units: the resident panel, device tables and small helpers.
 */
#ifndef GEPI_HOST_H
#define GEPI_HOST_H

#include <hip/hip_runtime.h>

#include <stddef.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "../../include/gepicount.h"
#include "gepi_device.h"
#include "gepi_internal.h"
#include "gepi_score.h"
#include "gepi_stage.h"

#define HIP_TRY(expr)                                                                     \
    do {                                                                                  \
        hipError_t e_ = (expr);                                                           \
        if (e_ != hipSuccess)                                                             \
            return gepi_fail(e_ == hipErrorOutOfMemory ? GEPI_ERR_NOMEM : GEPI_ERR_DEVICE, \
                             "%s failed: %s (%s:%d)", #expr, hipGetErrorString(e_),        \
                             __FILE__, __LINE__);                                         \
    } while (0)

namespace gepi_host {

using gepi::Cand;
using gepi::CompressWord;
using gepi::Pend;
using gepi::ScanState;

struct DeviceTables {
    int32_t tmax = -1;
    double *lhi = nullptr, *llo = nullptr, *lfact = nullptr;
};

} // namespace gepi_host

struct gepi_panel {
    using DeviceTables = gepi_host::DeviceTables;
    int device = 0;
    int64_t n_var = 0;
    int32_t n_samples = 0;
    int32_t w64 = 0;
    /* every valid call carries an allele (always so for .bed genotypes), so
     * that three genotypes describe it (count_f4g_unit)                    */
    bool three_genotypes = true;
    bool complete = false; /* no call of the panel is missing                */
    uint64_t *d_nat = nullptr;
    hipStream_t stream = nullptr;
    /* per-scan workspace, grown on demand and reused */
    uint32_t *d_cls = nullptr;
    size_t cls_bytes = 0;
    uint64_t *d_clsk = nullptr;
    size_t clsk_bytes = 0;
    int32_t *d_perm = nullptr;
    size_t perm_bytes = 0;
    gepi::CompressWord *d_cw = nullptr; /* fp4 path: class compression words */
    size_t cw_bytes = 0;
    gepi::PairRec *d_park = nullptr; /* fp4 wave tiles, Fisher: parked pairs */
    size_t park_bytes = 0;
    gepi::Cand *d_cand[2] = {nullptr, nullptr};
    gepi::Pend *d_pend = nullptr;
    unsigned long long buf_cap = 0;  /* records in the candidate buffer  */
    unsigned long long buf2_cap = 0; /* records in the second one        */
    size_t pend_bytes = 0;           /* pending list, then pairs put off  */
    gepi::ScanState *d_state = nullptr;
    uint64_t *d_small = nullptr;
    DeviceTables tabs;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    std::vector<hipEvent_t> band_ev; /* two per band of a planned scan: some from
                                      * the start, more as bands need them      */
    /* pinned, mapped: the band reports and small result lists the device
     * writes (HostMail) */
    void *mail = nullptr;
};


namespace gepi_host {

/* Makes `device` current; fails unless it is a gfx950. */
int set_device(int device);

/* Compute units of a device seen by set_device (256 if unknown). */
int32_t device_cus(int device);

/* Workgroups per CU of the persistent batched fp4 count launch (0: one
 * tile per workgroup); dflt unless GEPI_F4_WG_PER_CU overrides it. */
int f4_wg_per_cu(int dflt);

/* Grows the t*log2(t) and ln(t!) tables to cover t <= tmax. */
int ensure_tables(DeviceTables &tabs, int32_t tmax, hipStream_t stream);

template <typename T>
int grow(T **ptr, size_t *have, size_t need) {
    if (need <= *have && *ptr) return GEPI_OK;
    hipFree(*ptr);
    *ptr = nullptr;
    *have = 0;
    HIP_TRY(hipMalloc(ptr, need));
    *have = need;
    return GEPI_OK;
}


/* Coefficients of a lower bound of 1/g(p), p = min(y, z)/(y + z), over the
 * tables of a scan with classes of n0 and n1 samples (y <= n0, z <= n1):
 * 1/g(p) >= h0 + h1 min(y, z), the tangent of the convex 1/g at p0 =
 * min(n0, n1)/(n0 + n1) (g as in gepi_device.h's filter), less 1e-6 for the
 * roundings.                                                              */
inline void chi2_slope(int32_t n0, int32_t n1, float *h0, float *h1) {
    const double n = (double)n0 + n1, p = n > 0 ? std::min(n0, n1) / n : 0.0;
    double h = 1.0, d = 0.5; /* 1/g and its slope at p = 0 */
    if (p > 0.0) {
        const double l = -std::log1p(-p), g = l * (1.0 - p) / p;
        h = 1.0 / g;
        /* the difference loses digits for small p, where it nears 1/2 */
        d = p < 1e-4 ? 0.5 : (l / (p * p) - 1.0 / p) / (g * g);
    }
    *h0 = (float)(h - d * p - 1e-6);
    *h1 = n > 0 ? (float)(d / n * (1.0 - 1e-6)) : 0.0f;
}

/* The super-steps of a scan (384 samples of a class each, class 0 first)
 * in the panel's file order, for k_class_geno.                            */
inline void build_super_src(const std::vector<gepi::CompressWord> &cw, int32_t w64, int32_t n0,
                            int32_t n1, std::vector<gepi::SuperSrc> &src) {
    src.clear();
    const int32_t nw32 = 2 * w64;
    for (int c = 0; c < 2; c++) {
        const int32_t n = c == 0 ? n0 : n1;
        int32_t j = 0, seen = 0; /* class samples before word j */
        auto upto = [&](int32_t s) { /* word j holds class sample s */
            while (j < nw32 && seen + (int32_t)cw[(size_t)c * nw32 + j].cnt <= s)
                seen += (int32_t)cw[(size_t)c * nw32 + j++].cnt;
        };
        for (int32_t s = 0; s < n; s += 384) {
            gepi::SuperSrc r;
            r.cls = c;
            upto(s);
            r.j0 = j;
            r.skip = s - seen;
            upto(std::min(n, s + 384) - 1);
            r.j1 = j + 1;
            src.push_back(r);
        }
    }
}

/* The screen's constants of a scan (count_f4g_unit); g.miss is the caller's. */
inline void screen_consts(int32_t n0, int32_t n1, gepi::CountArgs &g) {
    const double n = (double)n0 + n1, p = n > 0 ? n0 / n : 0.5, s = std::min(p, 1.0 - p);
    /* k = (2 g(s) - 1) / s; a class without samples has no information (every
     * pair passes or none: both are right)                                 */
    const double k = s > 0.0 ? (2.0 * -std::log1p(-s) * (1.0 - s) / s - 1.0) / s * (1.0 + 1e-6) : 0.0;
    g.sc_p = (float)p;
    g.sc_k = (float)k;
    g.sc_q = (float)(2.0 * p * (1.0 - p) * (1.0 - 1e-4)); /* 1e-4: the roundings */
    g.sc_m = (float)(2.0 * p * (1.0 - p) * (1.0 - 1e-4) * n);
    /* counts up to n leave 24 - bits(n) bits for the fraction; at least 2^-12,
     * below which it no longer matters                                     */
    int bits = 0;
    while (bits < 16 && n >= (double)(1 << bits)) bits++;
    const double start = std::ldexp(1.0, -std::min(24 - bits, 12));
    g.sc_start = (float)start;
    g.sc_sub = (float)(18.0 * start * (1.0 + 2.0 * k) + 1e-3);
}

/* Whether the screen of the genotype table is near enough to spare the tests
 * that come after it: its k grows as 1/s with the smaller class's share s, and
 * k|u| with the spread of a cell's u, sqrt(s (1-s) / n).  Whole scans of 20,000
 * variants, top-100 and top-1,000, against the LDS-staged kernel's time (with
 * missing calls; without): entropy with 2,048 samples 0.79-0.82 at s = 0.1 (0.59-
 * 0.63), 0.94-1.04 at 0.05 (0.70-0.79), 1.35 at 0.03 (1.01-1.26), 2.3 at 0.015;
 * with 512 samples 1.01-1.05 at 0.2 (0.79-0.85), 1.13-1.17 at 0.1 (0.89-0.92),
 * 1.25-1.34 at 0.05; Fisher with 2,048 samples 0.86-1.07 at 0.2 (0.65-0.83),
 * 1.04-1.30 at 0.1 (0.83-1.03), 1.42-1.83 at 0.05, with 512 samples 1.10-1.40 at
 * 0.2 (0.97-1.17), 1.5-1.8 at 0.1.  Where it does not pay, the wave tiles run on
 * allele planes from F4W_MIN_KSTEPS K steps on (0.81-0.87 of the LDS-staged
 * kernel's time there with 2,048 samples).                                 */
inline bool screen_pays(int32_t n0, int32_t n1, bool fisher, bool complete) {
    const double n = (double)n0 + n1, s = n > 0 ? std::min(n0, n1) / n : 0.0;
    if (s <= 0.0) return true; /* nothing is associated: every pair passes any filter */
    const double k = (2.0 * -std::log1p(-s) * (1.0 - s) / s - 1.0) / s, spread = k * k * s * (1.0 - s) / n;
    if (fisher) return complete ? s >= 0.08 && spread <= 4e-3 : s >= 0.12 && spread <= 2.5e-3;
    return complete ? s >= 0.045 && spread <= 1.4e-2 : s >= 0.06 && spread <= 7e-3;
}

/* Records of the list of pairs that the count kernel puts off (48 bytes): one
 * for every 4 pairs of the scan (at 16 small scans with loose thresholds took
 * 1.12x the time: 1,020 x 89, 2,000 x 1,000), at most `most`, beyond which the
 * kernel tests its pairs itself, as it does where no list fits.  None from PAIRS_MAX_KSTEPS K steps on, where the other
 * workgroup of the CU fills the time of a test with its longer K loop: whole
 * scans of 20,000 variants, top-1,000, against tests in the kernel, took 0.90x
 * the time with 256 samples (Fisher 0.88x), 0.90x (0.89x) with 1,024, 0.92x
 * (0.92x) with 2,048, 0.98x (0.95x) with 4,096 and 1.00x (0.98x) with 8,192.  */
constexpr int PAIRS_WG_PER_CU = 8;
constexpr int64_t PAIRS_MOST = 1 << 22;       /* single scans: 201 MB          */
constexpr int64_t PAIRS_MOST_BATCH = 1 << 21; /* a scan of the engine: 101 MB  */
constexpr int32_t PAIRS_MAX_KSTEPS = 48;
constexpr size_t PAIR_BYTES = 48;
inline uint32_t pair_list_cap(int64_t n_tiles, int32_t ks, int64_t most) {
    if (ks > PAIRS_MAX_KSTEPS) return 0;
    /* test hook: at most so many records (0: as where the list does not fit) */
    if (const char *env = getenv("GEPI_PAIR_CAP")) most = std::min<int64_t>(most, std::max(atoll(env), 0ll));
    return (uint32_t)std::min<int64_t>(std::max<int64_t>(n_tiles * (64 * 32 / 4), 4096), most);
}

/* Units (two tiles) at the start of a band of n tiles under a guessed
 * threshold that test their pairs in the kernel, so that a guess far too
 * loose shows before the list of pairs has filled (band_full): none in a band
 * whose workgroups are all resident at once.                              */
inline int32_t pairs_from(int64_t n_tiles) { return n_tiles >= 2048 ? (int32_t)std::min<int64_t>(n_tiles / 512, 64) : 0; }

/* ---- planned bands --------------------------------------------------------
 * A scan's bands need no answer from the device between them: a band's
 * count, exact and top-k launches find the threshold, the lists and an
 * overflow flag in device memory, so all of them can be enqueued at once and
 * their reports read at the end (bands that overflowed are redone; the order
 * of bands does not change the result).  What has to be chosen beforehand is
 * the size of each band, from how many evaluations its threshold lets
 * through, and a threshold for the first one.
 *
 * Without association 2 m I (I in nats) of a table is close to chi-square
 * with one degree of freedom, and P(p <= a) of a Fisher test is at most a.
 * So the first band, a pilot, admits the quantile where GUESS times k of its
 * evaluations are expected: few enough to be cheap, and if the k best are
 * among them (nearly always: the count says so) the threshold was valid.
 * The others run under the k-th key so far.  A scan that ends with fewer than
 * k records is run again without the guess, and a band that finds far more
 * than expected stops and gives the threshold that it is redone under (room).  (Guessing the whole scan's
 * threshold after the pilot saved 10-15% where it held, but the tail hangs
 * on the few variants with the largest effects of their own: over seeds the
 * k-th key had 0.17 to 2 times the expected evaluations beyond it.)
 * Against bands that began with one tile admitting everything and grew
 * fourfold, a host round trip (40 us) and a selection between two: 1,024 x
 * 256 0.73 -> 0.13 ms (5 bands -> 1), 3,001 x 777 Fisher 1.44 -> 0.29, 20,000
 * x 2,048 3.69 -> 2.38 (10 -> 3), 8,000 x 20,001 3.84 -> 2.50.               */
constexpr double GUESS_ENTROPY = 7.5; /* 8: 1,024 x 256 top-100 selects for 54 us, 7.5: 47 */
/* Fisher: 16 for the 100 best, where a few variants decide, down to 4 for long
 * rankings, whose count varies less: each guessed evaluation that passes the
 * bound costs a walk over its tables (3,000 x 2,000 top-10,000 1.85 -> 0.7 ms,
 * 514 x 9,799 top-2,000 1.95 -> 0.75).                                      */
inline double guess_fisher(double k) { return std::max(4.0, std::min(16.0, 16.0 * std::cbrt(100.0 / k))); }
constexpr double LOOP_GUESS_ENTROPY = 2.0, LOOP_GUESS_FISHER = 4.0; /* long rankings */

/* P(chi2_1 > t) and its inverse */
inline double chi2_tail(double t) { return std::erfc(std::sqrt(0.5 * std::max(t, 0.0))); }
inline double chi2_quantile(double p) {
    double lo = 0.0, hi = 1400.0;
    for (int i = 0; i < 60; i++) {
        const double mid = 0.5 * (lo + hi);
        (chi2_tail(mid) > p ? lo : hi) = mid;
    }
    return lo;
}

/* The standard deviation of a 2 x 2 table's count with both margins fixed, the
 * function true for a tenth of the samples. */
inline double fisher_spread(int32_t n0, int32_t n1) {
    const double n = (double)n0 + n1;
    return n > 0 ? std::max(0.4, 0.3 * std::sqrt((double)n0 * n1 / n)) : 0.4;
}

struct BandPlan {
    bool entropy;
    double evals_tile;  /* evaluations per tile, on average: less than a whole
                         * tile's on small panels                             */
    double h;           /* chi-square coefficient per nat (chi2_slope)       */
    double sd;          /* Fisher: of a table's count (fisher_spread)        */
    double k;
    double most;        /* survivors a band may have                         */
    double c;           /* GUESS or LOOP_GUESS of the objective              */
    double factor = 1.0; /* survivors measured over survivors expected       */
    double spread = 16.0; /* survivors a list takes over those expected (room) */
    double walks = 65536; /* records scored in little more than one's time     */
    double limit = 1048576.0; /* tiles of one band at most (longest)           */

    /* Expected survivors of the chi-square bound per evaluation under the
     * threshold that admits a share q: its cut is h/2 of the quantile (a few
     * times fewer become records).  Fisher's check of log10 P(obs) passes what
     * is less probable than q: of a normal count with the spread sd, those
     * beyond z with the density phi(z) / sd = q, so all of them where sd q
     * nears phi(0): 4 times q for 2,048 samples and 2e-4, all for 46,000 and
     * 0.02.  (With 4 q, Fisher top-20,000 of 600 x 46,000 planned for a ninth of what
     * passed: 14.7 -> 36.2 ms.)                                             */
    double pass(double q) const {
        q = std::min(q, 1.0);
        if (entropy) return chi2_tail(0.5 * h * chi2_quantile(q));
        const double u = 2.5066283 * sd * q;
        return std::max(std::min(4.0 * q, 1.0), u < 1.0 ? chi2_tail(-2.0 * std::log(std::max(u, 1e-300))) : 1.0);
    }
    double survivors(int64_t tiles, double q) const {
        return factor * (double)tiles * evals_tile * pass(q);
    }
    /* the share of n tiles' evaluations that the first threshold admits */
    double share(int64_t n) const { return c * k / ((double)n * evals_tile); }
    /* the score that a share q of unassociated evaluations reaches */
    double score(double q, int32_t n) const {
        return entropy ? -chi2_quantile(q) / (2.0 * n) * 1.4426950408889634 : std::log10(q);
    }
    /* the first band: a scan of up to about 5,000 variants whole; else a pilot
     * of one tile per workgroup the chip holds, or more where that would
     * admit more than 4e-5 (the filter's expensive branch in most waves)   */
    int64_t first(int64_t n_tiles) const {
        if (n_tiles <= 6400 && survivors(n_tiles, share(n_tiles)) <= 600000.0) return n_tiles;
        return std::min<int64_t>(n_tiles, std::max<int64_t>(1024, (int64_t)(share(1) / 4e-5)));
    }
    /* whether a guess for n tiles tells anything and the lists hold it.  Of
     * entropy's survivors of the bound only those within a float's margin of
     * the threshold become records, 1.0-1.2 times the share aimed at (with
     * all of them counted, 1,024 x 256 top-1,000 ran four bands instead of one)  */
    double records(int64_t n) const { return entropy ? 1.5 * c * k : survivors(n, share(n)); }
    bool sound(int64_t n, unsigned long long cap) const {
        /* Fisher: a guess whose check passes a quarter of the evaluations tells
         * little; below, lists that turn out short cost little (room)      */
        return share(n) <= 0.1 && 1.5 * (c + 1.0) * k <= (double)cap &&
               records(n) <= (entropy ? most : 3.2 * most) && (entropy || pass(share(n)) <= 0.25);
    }
    /* Places that a planned band may fill in the pending list (of pcap):
     * `spread` times what is expected (unrelated phenotypes gave up to 8 times,
     * with rare alleles and uneven classes).  More of them means a threshold
     * far too loose: phenotypes that follow ancestry, linked or associated
     * variants, where nearly every evaluation may pass a guess made for
     * unrelated ones.  The rest of the band is left out (band_full), the
     * list's first `scored` records get their scores, the k-th key becomes the
     * threshold, and the band is redone in pieces.  Phenotypes that follow two
     * ancestries, against bands that grow from one tile without a guess and
     * against a guess with full lists: 20,000 x 2,048 entropy top-10,000 22.0
     * and 168.6 -> 3.6 ms, Fisher top-1,000 6.7 and 124.7 -> 4.5; 3,001 x 777
     * entropy top-100 1.17 and 12.6 -> 0.66, Fisher 1.44 and 18.3 -> 0.99; 4
     * scans of 5,000 x 1,000 batched, Fisher top-100, 3.7 and 31.0 -> 3.0.  */
    unsigned long long room(double expected, unsigned long long pcap) const {
        return std::min<unsigned long long>(pcap, (unsigned long long)std::max(65536.0, spread * expected));
    }
    uint32_t scored() const { return (uint32_t)std::min(walks / 4 + 8.0 * k, 4.0e9); }
    /* Redoing a band of n tiles after that: the k-th of `found` records lets
     * through a share of at most k / found, so its first tiles are as many as
     * pass `aim` evaluations then (at most a quarter: a band of one tile
     * always fits); the following ones grow fourfold with the threshold.   */
    double aim() const { return std::max(walks, 2.0 * k); }
    int64_t again(int64_t n, double found) const {
        const double tiles = aim() * std::max(1.0, found / k) / evals_tile;
        return std::max<int64_t>(1, std::min<int64_t>(n / 4, (int64_t)tiles));
    }
    unsigned long long room_again(unsigned long long pcap) const {
        return std::min<unsigned long long>(pcap, (unsigned long long)std::max(4.0 * aim(), gepi::TILE_EVALS_MAX + 1024.0));
    }
    /* Tiles of one band at most: a third of the scan (100,000 x 8,192
     * ran 1.5% slower with an eighth, 0.3-0.8% with a quarter, 0-0.5% so), or what
     * takes about 2 ms (0.7 ns for 64 x 32 pairs and 128 samples).  A few linked variants
     * late in a band can fill its list, and the time before that is lost: with
     * the last band as 85% of the scan, 40,000 x 4,096 in linked blocks, five
     * of them with an effect, entropy top-100, took 20.5 ms and 15.8 now (16.1
     * in bands that grow without a guess).                                  */
    static double longest(int64_t n_tiles, int64_t n_ks) {
        return std::min(1048576.0, std::max((double)n_tiles / 3, 3.0e6 / (double)std::max<int64_t>(1, n_ks)));
    }
    /* the threshold that lets through what is expected after `done` tiles */
    double share_after(int64_t done) const { return 1.3 * k / ((double)done * evals_tile); }
    /* survivors found in n tiles under the threshold that admits a share q */
    void learn(int64_t n, double q, unsigned long long found) {
        factor = 1.0;
        factor = std::min(64.0, std::max(0.25, (double)found / std::max(1.0, survivors(n, q))));
    }
    /* Tiles of the band that follows `done` tiles.  About 250,000 survivors
     * cost what a band's fixed part does (100 us); at least three times what
     * is done while the list holds them, at most that for Fisher and eight
     * times for entropy (the pairs that pass the screen cost more under an
     * older threshold).                                                     */
    int64_t next(int64_t done, int64_t left) const {
        const double per = survivors(1, share_after(done));
        const double cheap = std::min(std::max(250000.0 / per, 3.0 * (double)done),
                                      (entropy ? 8.0 : 3.0) * (double)done);
        const double tiles = std::min({cheap, most / per, limit, (double)left});
        /* a remainder below a fifth of the band goes with it */
        if ((double)left < 1.2 * tiles && (double)left * per < most) return left;
        return std::max<int64_t>(1, (int64_t)tiles);
    }
};

/* The first n records as results. */
inline int64_t results_of(const gepi::Cand *rec, int64_t n, gepi_result *tops) {
    for (int64_t i = 0; i < n; i++) {
        const gepi::Cand &c = rec[i];
        gepi_result &r = tops[i];
        r.sA = (int64_t)(c.idx >> 32);
        r.sB = (int64_t)((c.idx >> 3) & 0x1FFFFFFFull);
        r.fun = (int32_t)(c.idx & 7);
        r.w = (int32_t)c.w;
        r.x = (int32_t)c.x;
        r.y = (int32_t)c.y;
        r.z = (int32_t)c.z;
        r.obj = c.score;
        r.reserved = 0;
    }
    return n;
}

/* Sorts candidate records by the canonical key and writes the first
 * min(k, size) as results; returns how many were written.                   */
inline int64_t candidates_to_results(std::vector<gepi::Cand> &host, int64_t k, gepi_result *tops) {
    std::sort(host.begin(), host.end(), [](const gepi::Cand &a, const gepi::Cand &b) {
        const uint64_t ha = gepi::order_bits(a.score), hb = gepi::order_bits(b.score);
        return ha < hb || (ha == hb && a.idx < b.idx);
    });
    return results_of(host.data(), std::min<int64_t>((int64_t)host.size(), k), tops);
}

/* Class compression words of a scan: [2][2 * w64], class 0 then class 1;
 * mask bits at or beyond n_samples are dropped.  Returns (n0, n1).          */
inline void build_compress_words(const uint64_t *mask_ctrl, const uint64_t *mask_case,
                                 int32_t n_samples, int32_t w64,
                                 std::vector<gepi::CompressWord> &cw, int32_t &n0, int32_t &n1) {
    const int32_t nw32 = 2 * w64;
    cw.resize((size_t)2 * std::max(nw32, 1));
    int32_t cnt[2] = {0, 0};
    for (int c = 0; c < 2; c++) {
        const uint64_t *mk = c == 0 ? mask_ctrl : mask_case;
        for (int32_t j = 0; j < nw32; j++) {
            uint32_t m = 0;
            if (mk) m = (uint32_t)(mk[j >> 1] >> (32 * (j & 1)));
            const int32_t lo = 32 * j;
            if (lo >= n_samples)
                m = 0;
            else if (n_samples - lo < 32)
                m &= (1u << (n_samples - lo)) - 1u;
            cw[(size_t)c * nw32 + j] = gepi::make_compress_word(m);
            cnt[c] += (int32_t)cw[(size_t)c * nw32 + j].cnt;
        }
    }
    n0 = cnt[0];
    n1 = cnt[1];
}

} // namespace gepi_host

#endif
