"""What a user of the framework has it do, as cases that can be timed and compared.

listed() holds twelve cases from the smallest call to the largest, draw(rng) more of
the same ranges; prepare() makes what a program has in hand before the call (genotypes
and phenotypes from a seed, a resident panel, an engine, a server), run() is one pass
through the public entry points, and exact() gives the scores of the best evaluations
in 64-bit torch arithmetic without the framework.

Sizes are those of the synthetic workloads (1,024 x 256, 20,000 x 2,048, 100,000 x
8,192, the mix of uneven scans, the re-scanned resident panel), of the reader's test
data (1,020 x 89), or generic odd ones.  Genotypes are Hardy-Weinberg draws with the
workloads' allele frequencies and missing rates; phenotypes are unrelated to them,
as in the workloads, so a ranking is the tail of many near-independent pairs.
"""
import math

import numpy as np
import torch

import gepicount_amd as ge
from gepicount_amd import api, synth

ENTROPY, FISHER = 0, 1
DEV = "cuda"
FIELDS = ("sA", "sB", "w", "x", "y", "z", "obj", "fun")


def listed():
    return [
        # The drop-in call on reader planes at the size of the reader's test data: a whole
        # process_gpu_1 (upload, scan, release), where latency is everything.
        dict(name="thin_dropin", kind="dropin", n_var=1020, n=89, case_frac=0.5, out_frac=0.0,
             maf="uniform", miss=0.006, ffun=ENTROPY, topk=1000),
        # The small workload on a resident panel: the smallest scan of a serving program.
        dict(name="small_entropy", kind="scan", n_var=1024, n=256, case_frac=0.5, out_frac=0.0,
             maf="uniform", miss=0.0, ffun=ENTROPY, topk=100),
        # A candidate-gene panel with odd sizes, uneven classes and samples left out, Fisher.
        dict(name="odd_fisher", kind="scan", n_var=3001, n=777, case_frac=0.37, out_frac=0.05,
             maf="uniform", miss=0.01, ffun=FISHER, topk=100),
        # The medium workload, entropy: an ordinary scan.
        dict(name="medium_entropy", kind="scan", n_var=20000, n=2048, case_frac=0.5, out_frac=0.0,
             maf="uniform", miss=0.01, ffun=ENTROPY, topk=1000),
        # The same with the Fisher objective.
        dict(name="medium_fisher", kind="scan", n_var=20000, n=2048, case_frac=0.5, out_frac=0.0,
             maf="uniform", miss=0.01, ffun=FISHER, topk=1000),
        # The command line's default: the drop-in call with -N at its default of 1,000,000.
        dict(name="medium_default_n", kind="dropin", n_var=20000, n=2048, case_frac=0.5,
             out_frac=0.0, maf="uniform", miss=0.01, ffun=ENTROPY, topk=1000000),
        # An imputed panel (no missing calls), odd sizes.
        dict(name="imputed_entropy", kind="scan", n_var=30001, n=3001, case_frac=0.4, out_frac=0.0,
             maf="beta", miss=0.0, ffun=ENTROPY, topk=1000),
        # More samples than the reference accepts: few variants, a biobank's samples.
        dict(name="wide_entropy", kind="scan", n_var=8000, n=20001, case_frac=0.3, out_frac=0.0,
             maf="beta", miss=0.02, ffun=ENTROPY, topk=1000),
        # The large workload: the framework's headline.
        dict(name="large_entropy", kind="scan", n_var=100000, n=8192, case_frac=0.3, out_frac=0.0,
             maf="beta", miss=0.02, ffun=ENTROPY, topk=10000),
        # Many uneven scans at once through the batch engine, every fourth with Fisher.
        dict(name="batch_mix", kind="batch", scans=24, mix_seed=1004),
        # A server with a resident panel that is scanned again with new phenotypes, and
        # uneven scans beside it: all requests submitted, then waited for.
        dict(name="serve_rescans", kind="serve", n_var=12000, n=4000, rescans=6, scans=10,
             mix_seed=77),
        # Quality control before a scan: .bed bytes to the device, missing counts per
        # variant and sample, the filtered panel.
        dict(name="ingest_qa", kind="ingest", n_var=50000, n=4000, maf="uniform", miss=0.02),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["scan", "scan", "scan", "scan", "dropin", "noalloc", "batch", "serve",
                       "ingest"])
    if kind == "batch":
        return dict(kind=kind, scans=rng.randint(2, 24), mix_seed=rng.randint(1, 10 ** 6))
    if kind == "serve":
        return dict(kind=kind, n_var=_log_int(rng, 500, 12000), n=_log_int(rng, 200, 4000),
                    rescans=rng.randint(1, 6), scans=rng.randint(0, 8),
                    mix_seed=rng.randint(1, 10 ** 6))
    if kind == "ingest":
        return dict(kind=kind, n_var=_log_int(rng, 500, 50000), n=_log_int(rng, 64, 4000),
                    maf=rng.choice(["uniform", "beta"]), miss=rng.choice([0.005, 0.02, 0.04]))
    # samples over the whole range, variants so that a scan stays under a quarter of
    # the largest listed one
    n = _log_int(rng, 64, 20001)
    top = {"scan": 60000, "dropin": 15000, "noalloc": 4000}[kind]
    n_var = _log_int(rng, 500, max(501, min(top, int(math.sqrt(2.0e13 / n)))))
    most = {"scan": 200000, "dropin": 1000000, "noalloc": 20000}[kind]
    if kind == "noalloc":
        n = min(n, 6000)
    return dict(kind=kind, n_var=n_var, n=n, case_frac=round(rng.uniform(0.2, 0.8), 3),
                out_frac=rng.choice([0.0, 0.0, 0.05]), maf=rng.choice(["uniform", "beta"]),
                miss=rng.choice([0.0, 0.005, 0.01, 0.02]), ffun=rng.choice([ENTROPY, ENTROPY, FISHER]),
                topk=_log_int(rng, 10, most))


# ---- inputs ------------------------------------------------------------------------


def _codes(gen, n_var, n, maf, miss, spread=False):
    """PLINK codes [n_var][n] uint8 on the GPU, a chunk of variants at a time: yields (first, codes).
    spread: missing rates that differ from variant to variant, with `miss` as their mean."""
    u = torch.rand(n_var, generator=gen, device=DEV)
    if maf == "beta":
        # Beta(0.5, 2), the large workload's skew towards rare alleles, by its inverse:
        # F(x) = 1.5 s - 0.5 s^3 with s = sqrt(x) = 2 sin(asin(u) / 3)
        f = (4.0 * torch.sin(torch.asin(u) / 3.0) ** 2).clamp(0.01, 0.5)
    else:
        f = 0.01 + 0.49 * u
    m = torch.full((n_var,), float(miss), device=DEV)
    if spread:
        m = -float(miss) * torch.log1p(-torch.rand(n_var, generator=gen, device=DEV))
    step = max(64, (1 << 25) // max(n, 1))
    for v0 in range(0, n_var, step):
        fc, mc = f[v0:v0 + step, None], m[v0:v0 + step, None]
        shape = (fc.shape[0], n)
        g = (torch.rand(shape, generator=gen, device=DEV) < fc).to(torch.uint8)
        g += (torch.rand(shape, generator=gen, device=DEV) < fc).to(torch.uint8)
        c = 3 - g  # 0 copies -> 3, 1 -> 2, 2 -> 0
        c[g == 2] = 0
        if miss > 0:
            c[torch.rand(shape, generator=gen, device=DEV) < mc] = 1
        yield v0, c


def _payload(gen, n_var, n, maf, miss, spread=False):
    n4 = (n + 3) // 4
    out = np.empty((n_var, n4), np.uint8)
    for v0, c in _codes(gen, n_var, n, maf, miss, spread):
        c = torch.nn.functional.pad(c, (0, 4 * n4 - n)).view(c.shape[0], n4, 4)
        b = c[:, :, 0] | (c[:, :, 1] << 2) | (c[:, :, 2] << 4) | (c[:, :, 3] << 6)
        out[v0:v0 + b.shape[0]] = b.cpu().numpy()
    return out


def _pack_bits(m):
    """Bool [r][n] -> uint64 [r][ceil(n / 64)], bit s of a row = sample s."""
    r, n = m.shape
    w = (n + 63) // 64
    m = torch.nn.functional.pad(m.to(torch.uint8), (0, 64 * w - n)).view(r, 8 * w, 8)
    b = m[:, :, 0].clone()
    for i in range(1, 8):
        b |= m[:, :, i] << i
    return b.cpu().numpy().view(np.uint64).reshape(r, w)


def _planes(gen, n_var, n, maf, miss):
    """Reader planes: rows 2i and 2i + 1 are the alleles of variant i."""
    w = (n + 63) // 64
    bits = np.empty((2 * n_var, w), np.uint64)
    valid = np.empty((2 * n_var, w), np.uint64)
    for v0, c in _codes(gen, n_var, n, maf, miss):
        r = slice(2 * v0, 2 * (v0 + c.shape[0]))
        bits[r][0::2] = _pack_bits((c == 0) | (c == 2))
        bits[r][1::2] = _pack_bits((c == 2) | (c == 3))
        valid[r][0::2] = _pack_bits(c != 1)
        valid[r][1::2] = valid[r][0::2]
    return bits, valid


def _pheno(rng, n, case_frac, out_frac=0.0):
    """1 control, 2 case, 0 left out."""
    p = np.ones(n, np.int64)
    order = rng.permutation(n)
    cases = max(1, int(round(case_frac * n)))
    p[order[:cases]] = 2
    if out_frac:
        p[rng.permutation(n)[:int(out_frac * n)]] = 0
    return p


def _gen(seed, k=0):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 1000 + k)


def _mix(case):
    """Sizes of a case's uneven scans (the mix workload's distributions, its smaller half)."""
    specs = synth.mix_specs(case["scans"], case["mix_seed"])
    for i, s in enumerate(specs):
        if case["kind"] == "serve":
            s["n_var"] = max(500, s["n_var"] // 4)
        s["ffun"] = FISHER if case["kind"] == "batch" and i % 4 == 3 else ENTROPY
    return specs


def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.Generator(np.random.PCG64(seed))
    if kind == "ingest":
        return dict(kind=kind, payload=_payload(_gen(seed), case["n_var"], case["n"], case["maf"],
                                                case["miss"], spread=True),
                    n_var=case["n_var"], n=case["n"])
    if kind == "batch":
        items = []
        for i, s in enumerate(_mix(case)):
            m0, m1 = synth.masks_from_pheno(_pheno(rng, s["n_samples"], s["n_case"] / s["n_samples"]))
            p = ge.Panel.from_bed(_payload(_gen(seed, i), s["n_var"], s["n_samples"], "uniform",
                                           s["miss"]), s["n_var"], s["n_samples"])
            items.append(dict(panel=p, mask_ctrl=m0, mask_case=m1, topmost=s["topk"], ffun=s["ffun"]))
        return dict(kind=kind, engine=ge.Engine(), items=items)
    if kind == "serve":
        server, asks = ge.Server(), []
        pid = server.add_panel_bed(_payload(_gen(seed, 999), case["n_var"], case["n"], "uniform", 0.01),
                                   case["n_var"], case["n"])
        for i in range(case["rescans"]):
            m0, m1 = synth.masks_from_pheno(_pheno(rng, case["n"], 0.3 + 0.05 * i))
            asks.append((pid, m0, m1))
        for i, s in enumerate(_mix(case)):
            m0, m1 = synth.masks_from_pheno(_pheno(rng, s["n_samples"], s["n_case"] / s["n_samples"]))
            q = server.add_panel_bed(_payload(_gen(seed, i), s["n_var"], s["n_samples"], "uniform",
                                              s["miss"]), s["n_var"], s["n_samples"])
            asks.append((q, m0, m1))
        return dict(kind=kind, server=server, asks=asks)
    m0, m1 = synth.masks_from_pheno(_pheno(rng, case["n"], case["case_frac"], case["out_frac"]))
    st = dict(kind=kind, m0=m0, m1=m1, n=case["n"], topk=case["topk"], ffun=case["ffun"])
    if kind == "dropin":
        st["bits"], st["valid"] = _planes(_gen(seed), case["n_var"], case["n"], case["maf"],
                                          case["miss"])
    else:
        st["panel"] = ge.Panel.from_bed(_payload(_gen(seed), case["n_var"], case["n"], case["maf"],
                                                 case["miss"]), case["n_var"], case["n"])
    return st


# ---- one pass ------------------------------------------------------------------------


def _fields(r):
    return {k: r[k] for k in FIELDS}


def run(st):
    kind = st["kind"]
    if kind == "scan":
        r, _ = st["panel"].scan(st["m0"], st["m1"], topmost=st["topk"], ffun=st["ffun"])
        return _fields(r)
    if kind == "noalloc":
        r, _ = st["panel"].scan_noalloc(st["m0"], st["m1"], topmost=st["topk"], ffun=st["ffun"])
        return _fields(r)
    if kind == "dropin":
        r, _ = api.process_gpu_1(st["bits"], st["valid"], st["m0"], st["m1"], st["n"],
                                 topmost=st["topk"], ffun=st["ffun"])
        return _fields(r)
    if kind == "batch":
        res, _ = st["engine"].scan_batch(st["items"])
        return dict(_fields(np.concatenate([r for r, _, _ in res])),
                    status=np.array([s for _, _, s in res]))
    if kind == "serve":
        tickets = [st["server"].submit(p, m0, m1, topmost=100) for p, m0, m1 in st["asks"]]
        res = [st["server"].wait(t) for t in tickets]
        return dict(_fields(np.concatenate([r for r, _, _ in res])),
                    status=np.array([s for _, _, s in res]))
    panel = ge.Panel.from_bed(st["payload"], st["n_var"], st["n"])
    vm, sm, bad_v, bad_s = panel.qa()
    kept, idx, keep = panel.filter()
    kept.close()
    panel.close()
    conforming = np.zeros(st["n_var"], np.bool_)
    conforming[idx] = True
    return dict(variant_missing=vm, sample_missing=sm, bad_variants=bad_v, bad_samples=bad_s,
                conforming=conforming, keep_samples=keep.view(np.int64))


# ---- what a pass cannot do without ----------------------------------------------------


def _scan_work(n_var, n, miss, topk):
    """Genotypes at 2 bits and the masks in, 48-byte results out; per variant pair and
    sample a multiply-add for each of the nine plane products (four without missing
    calls: the others are the variants' own counts)."""
    evals = 5 * n_var * (2 * n_var + 1)
    flops = 2.0 * (9 if miss > 0 else 4) * n * (n_var * (n_var + 1) / 2.0)
    return n_var * ((n + 3) // 4) + 2 * ((n + 7) // 8) + 48 * min(topk, evals), flops


def work(case):
    kind = case["kind"]
    if kind == "ingest":
        # .bed bytes read; the planes of the panel and of the filtered one written
        return dict(bytes=case["n_var"] * (((case["n"] + 3) // 4) + 2 * 3 * ((case["n"] + 63) // 64) * 8),
                    flops=0)
    if kind in ("batch", "serve"):
        b = f = 0.0
        parts = [(s["n_var"], s["n_samples"], s["miss"], 100) for s in _mix(case)]
        if kind == "serve":
            parts += [(case["n_var"], case["n"], 0.01, 100)] * case["rescans"]
        for p in parts:
            x, y = _scan_work(*p)
            b, f = b + x, f + y
        return dict(bytes=b, flops=f)
    b, f = _scan_work(case["n_var"], case["n"], case["miss"], case["topk"])
    if kind == "dropin":
        # reader planes: two allele rows and their valid bits a variant
        b += case["n_var"] * (4 * ((case["n"] + 63) // 64) * 8 - (case["n"] + 3) // 4)
    return dict(bytes=b, flops=f)


# ---- the scores in 64 bits --------------------------------------------------------------

EXACT_EVALS = 3.0e10


def _xlog2(n):
    t = torch.arange(n + 1, dtype=torch.float64, device=DEV)
    return torch.special.xlogy(t, t) / math.log(2.0)


def _fisher_p(w, x, y, z, lf):
    """log10 of the two-sided p of [[w, y-w], [x, z-x]], terms within 1e-7 of the observed."""
    w, x, y, z = (t.to(torch.int64) for t in (w, x, y, z))
    out = torch.zeros(w.shape, dtype=torch.float64, device=DEV)
    r, m = w + x, y + z
    most = int(torch.minimum(y, r).max()) + 1 if w.numel() else 1
    step = max(1, (1 << 24) // most)
    for i in range(0, w.numel(), step):
        s = slice(i, i + step)
        a = torch.arange(most, device=DEV)[None, :]
        ys, zs, rs, ms = (t[s, None] for t in (y, z, r, m))
        ok = (a <= ys) & (a <= rs) & (rs - a <= zs)
        ac = torch.where(ok, a, torch.zeros_like(a) + (rs - zs).clamp(min=0))
        lp = lf[ys] - lf[ac] - lf[ys - ac] + lf[zs] - lf[rs - ac] - lf[zs - rs + ac]
        lp = torch.where(ok, lp, torch.full_like(lp, -math.inf))
        obs = lp.gather(1, w[s, None])
        tail = torch.where(lp <= obs + 1e-7, lp, torch.full_like(lp, -math.inf))
        p = torch.logsumexp(tail, 1) - torch.logsumexp(lp, 1)
        out[s] = torch.where((tail == -math.inf).eq(lp == -math.inf).all(1), torch.zeros_like(p), p)
    return out / math.log(10.0)


def _exact_scan(chunks, n_var, pheno, ffun, topk):
    """The topk best scores, ascending, by brute force in blocks of variants."""
    n = len(pheno)
    codes = torch.empty((n_var, n), dtype=torch.uint8, device=DEV)
    for v0, c in chunks:
        codes[v0:v0 + c.shape[0]] = c
    ph = torch.from_numpy(pheno).to(DEV)
    planes = []
    for cls in (1, 2):
        c = codes[:, ph == cls]
        planes.append([p.to(torch.float32) for p in ((c == 0) | (c == 2), (c == 2) | (c == 3), c != 1)])
    lg = _xlog2(n + 1)
    t = torch.arange(n + 2, dtype=torch.float64, device=DEV)
    lf = torch.lgamma(t + 1.0)
    best = torch.empty(0, dtype=torch.float64, device=DEV)
    lim = math.inf
    block = max(1, min(n_var, (1 << 24) // n_var))
    for a0 in range(0, n_var, block):
        a1 = min(n_var, a0 + block)
        # c[class][p][q]: products of plane p of the block and plane q of variants up to it
        c = [[[pl[p][a0:a1] @ pl[q][:a1].T for q in range(3)] for p in range(3)] for pl in planes]
        va = torch.arange(a0, a1, device=DEV)[:, None]
        vb = torch.arange(a1, device=DEV)[None, :]
        y, z = (c[k][2][2].round().to(torch.int32) for k in (0, 1))
        for ia in (0, 1):
            for ib in (0, 1):
                real = (vb < va) | ((vb == va) & (ib <= ia))
                for f in range(5):
                    o = []
                    for k in (0, 1):
                        n11, na, nb, v = c[k][ia][ib], c[k][ia][2], c[k][2][ib], c[k][2][2]
                        o.append((n11, nb - n11, na - n11, v - na - nb + n11, na + nb - 2 * n11)[f]
                                 .round().to(torch.int32))
                    w, x = o
                    if ffun == ENTROPY:
                        m, r = y + z, w + x
                        s = lg[y] + lg[z] + lg[r] + lg[m - r] - lg[w] - lg[y - w] - lg[x] - lg[z - x] - lg[m]
                        s = torch.where(m > 0, s / m.clamp(min=1), torch.zeros_like(s))
                        s = s[real & (s <= lim)]
                    else:
                        m, r = y + z, w + x
                        lp = lf[y] + lf[z] + lf[r] + lf[m - r] - lf[w] - lf[y - w] - lf[x] - lf[z - x] - lf[m]
                        # p is at least the observed table's probability
                        at = real & (lp / math.log(10.0) <= lim + 1e-9)
                        if lim == math.inf and int(at.sum()) > 4 * topk + 4096:
                            first = torch.kthvalue(lp[at], 4 * topk + 4096).values
                            kept = at & (lp <= first)
                            s0 = _fisher_p(w[kept], x[kept], y[kept], z[kept], lf)
                            lim = float(torch.kthvalue(s0, min(topk, s0.numel())).values)
                            at = real & (lp / math.log(10.0) <= lim + 1e-9)
                        s = _fisher_p(w[at], x[at], y[at], z[at], lf)
                        s = s[s <= lim]
                    best = torch.cat([best, s])
                    if best.numel() > 4 * topk + (1 << 22) or (best.numel() > topk and f == 4):
                        best = torch.sort(best).values[:topk]
                        lim = float(best[-1]) if best.numel() == topk else math.inf
    return torch.sort(best).values[:topk].clamp(max=0.0)


def exact(case, seed):
    kind = case["kind"]
    if kind == "ingest":
        return None
    if kind in ("scan", "noalloc", "dropin"):
        evals = 5 * case["n_var"] * (2 * case["n_var"] + 1)
        if evals > EXACT_EVALS:
            return None
        rng = np.random.Generator(np.random.PCG64(seed))
        pheno = _pheno(rng, case["n"], case["case_frac"], case["out_frac"])
        obj = _exact_scan(_codes(_gen(seed), case["n_var"], case["n"], case["maf"], case["miss"]),
                          case["n_var"], pheno, case["ffun"], min(case["topk"], evals))
        return dict({k: None for k in FIELDS}, obj=obj.cpu().numpy())
    specs = _mix(case)
    total = sum(5 * s["n_var"] * (2 * s["n_var"] + 1) for s in specs)
    if total > EXACT_EVALS:
        return None
    rng = np.random.Generator(np.random.PCG64(seed))
    parts = []
    if kind == "serve":
        evals = 5 * case["n_var"] * (2 * case["n_var"] + 1)
        if total + evals * case["rescans"] > EXACT_EVALS:
            return None
        for i in range(case["rescans"]):
            ph = _pheno(rng, case["n"], 0.3 + 0.05 * i)
            parts.append(_exact_scan(_codes(_gen(seed, 999), case["n_var"], case["n"], "uniform", 0.01),
                                     case["n_var"], ph, ENTROPY, min(100, evals)))
    for i, s in enumerate(specs):
        ph = _pheno(rng, s["n_samples"], s["n_case"] / s["n_samples"])
        parts.append(_exact_scan(_codes(_gen(seed, i), s["n_var"], s["n_samples"], "uniform", s["miss"]),
                                 s["n_var"], ph, s["ffun"],
                                 min(100, 5 * s["n_var"] * (2 * s["n_var"] + 1))))
    return dict({k: None for k in FIELDS}, obj=torch.cat(parts).cpu().numpy(), status=None)
