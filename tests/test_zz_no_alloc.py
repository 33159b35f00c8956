"""gepi_scan_noalloc: the scan of a resident panel with every buffer in the
library's fixed per-GPU scratch array (no device allocation).  Results must
equal gepi_scan's bit for bit, on consecutive calls that reuse the array
with a smaller input second, and the call must not change the device's free
memory."""
import numpy as np
import pytest

import gepicount_amd as ge
from gepicount_amd import synth
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

FIELDS = ("sA", "sB", "fun", "w", "x", "y", "z", "obj")


def assert_same(got, ref, label):
    assert len(got) == len(ref), (label, len(got), len(ref))
    for k in FIELDS:
        if not np.array_equal(got[k], ref[k]):
            bad = int(np.flatnonzero(got[k] != ref[k])[0])
            raise AssertionError("%s: field %s differs first at rank %d: got %r ref %r" % (
                label, k, bad, got[bad], ref[bad]))


def free_bytes():
    """Free device memory from the HIP runtime the library itself uses."""
    import ctypes
    ge.lib()
    hip = ctypes.CDLL("libamdhip64.so.7")  # already loaded by the library
    free, total = ctypes.c_size_t(0), ctypes.c_size_t(0)
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_noalloc_equals_scan_on_consecutive_calls():
    print("case noalloc: 6000 x 2048 then 300 x 700", flush=True)
    big = synth.make_panel("medium", n_var=6000)
    small = synth.make_panel(spec=dict(n_var=300, n_samples=700, n_case=310,
                                       maf=("uniform", 0.01, 0.5), miss=0.02, planted=0, seed=77))
    # a scan on another panel first, so that the runtime's own lazily created
    # resources (staging buffers, module state) exist before free memory is read
    with ge.Panel.from_bed(small["payload"], small["n_var"], small["n_samples"]) as warm:
        m0, m1 = synth.masks_from_pheno(small["pheno"])
        warm.scan(m0, m1, topmost=10)
        warm.scan_noalloc(m0, m1, topmost=10)
    cases = [(big, 1000, 0), (big, 300, 1), (small, 200, 0), (small, 5000, 1)]
    for i, (p, k, ffun) in enumerate(cases):
        m0, m1 = synth.masks_from_pheno(p["pheno"])
        with ge.Panel.from_bed(p["payload"], p["n_var"], p["n_samples"]) as h:
            got, st = h.scan_noalloc(m0, m1, topmost=k, ffun=ffun)
            # the fp4 kernel chosen by objective and size: wave tiles for
            # entropy scans of at least 10 K steps of 128 samples
            ks = -(-st["n_class0"] // 128) - (-st["n_class1"] // 128)
            assert st["count_path"] == (3 if ffun == 0 and ks >= 10 else 4), st
            assert st["bytes_allocated"] == 0, st
            ref, st_ref = h.scan(m0, m1, topmost=k, ffun=ffun)
            assert st_ref["bytes_allocated"] > 0, "a fresh panel's first scan grows its workspace"
            assert_same(got, ref, "case %d vs gepi_scan" % i)
            # a repeated call: the runtime's own lazily created resources
            # exist by now, so free device memory must not move at all
            before = free_bytes()
            again, st2 = h.scan_noalloc(m0, m1, topmost=k, ffun=ffun)
            after = free_bytes()
            assert before == after, ("free memory changed", i, before, after)
            assert st2["bytes_allocated"] == 0
            assert_same(again, ref, "case %d repeated" % i)
    # the smaller panel also against the oracle
    m0, m1 = synth.masks_from_pheno(small["pheno"])
    with ge.Panel.from_bed(small["payload"], small["n_var"], small["n_samples"]) as h:
        got, _ = h.scan_noalloc(m0, m1, topmost=500)
        bits, valid = h.download()
    ref = orc.gold_scan(orc.Panel(bits, valid, m0, m1, small["n_samples"]), 500)
    assert_same(got, ref, "small vs oracle")


def test_noalloc_rejects_what_does_not_fit():
    print("case noalloc limits", flush=True)
    rng = np.random.default_rng(5)
    n_var, n = 100000, 2048
    payload = rng.integers(0, 256, size=(n_var, n // 4), dtype=np.uint8)
    pheno = synth.pheno_for(n, 1024, 9)
    m0, m1 = synth.masks_from_pheno(pheno)
    with ge.Panel.from_bed(payload, n_var, n) as h:
        with pytest.raises(ge.GepiError) as e:
            h.scan_noalloc(m0, m1, topmost=100)
        assert e.value.code == -3  # GEPI_ERR_LIMIT
        assert "scratch" in str(e.value)
    small = synth.make_panel("small", n_var=40)
    m0, m1 = synth.masks_from_pheno(small["pheno"])
    with ge.Panel.from_bed(small["payload"], small["n_var"], small["n_samples"]) as h:
        with pytest.raises(ge.GepiError) as e:
            h.scan_noalloc(m0, m1, topmost=100, count_path=2)
        assert e.value.code == -1 and "fp4" in str(e.value)  # GEPI_ERR_ARG
        # the array is usable after a rejected call
        got, _ = h.scan_noalloc(m0, m1, topmost=100)
        ref, _ = h.scan(m0, m1, topmost=100)
        assert_same(got, ref, "after rejection")


def fresh_panels(count):
    """Panels that no scan has run on, each with its stream, and masks for them;
    the library's kernels and scratch array have been used before."""
    p = synth.make_panel(spec=dict(n_var=300, n_samples=700, n_case=310, maf=("uniform", 0.01, 0.5),
                                   miss=0.02, planted=0, seed=78))
    m0, m1 = synth.masks_from_pheno(p["pheno"])
    made = [ge.Panel.from_bed(p["payload"], p["n_var"], p["n_samples"]) for _ in range(count + 1)]
    for k, ffun in ((50, 0), (6000, 0), (3000, 1)):
        made[0].scan_noalloc(m0, m1, topmost=k, ffun=ffun)
    made.pop(0).close()
    return made, m0, m1


def test_noalloc_first_calls_leave_device_memory():
    """Kernels that need private memory have the runtime allocate it for a
    queue's first one: more panels than there are hardware queues, short and
    sorted rankings, both objectives."""
    print("case noalloc first calls", flush=True)
    panels, m0, m1 = fresh_panels(8)
    for h in panels:
        for k, ffun in ((50, 0), (6000, 0), (3000, 1)):
            before = free_bytes()
            h.scan_noalloc(m0, m1, topmost=k, ffun=ffun)
            assert free_bytes() == before, (k, ffun)
    for h in panels:
        h.close()


def test_noalloc_first_calls_map_nothing():
    """Device and pinned host memory that the runtime hands out is mapped from
    the render node: a panel's first scans map none."""
    print("case noalloc mappings", flush=True)

    def mapped():
        with open("/proc/self/maps") as f:
            return {line.split()[0] for line in f if "/dev/dri/" in line}

    panels, m0, m1 = fresh_panels(3)
    for h in panels:
        for k, ffun in ((50, 0), (6000, 0), (3000, 1)):
            before = mapped()
            _, st = h.scan_noalloc(m0, m1, topmost=k, ffun=ffun)
            assert mapped() <= before, (k, ffun)
            assert st["bytes_allocated"] == 0
    for h in panels:
        h.close()


def test_noalloc_longest_ranking():
    """The scratch array holds as long a ranking of a panel on genotype planes as
    of one on allele planes (a valid call without an allele): the places of its
    super-steps take none of it.  The longest that the second one's message
    leaves room for, and one more."""
    print("case noalloc longest ranking", flush=True)
    n_var, n = 400, 40000
    rng = np.random.default_rng(79)
    codes = rng.choice(np.array([0, 2, 3], np.uint8), size=(n_var, n))
    bits, valid = orc.planes_from_codes(codes)
    m0, m1 = orc.masks_from_classes(np.arange(n) % 2)
    bare = bits.copy()
    bare[0:2, 0] = 0
    with ge.Panel.from_planes(bare, valid, n) as h:
        with pytest.raises(ge.GepiError) as e:
            h.scan_noalloc(m0, m1, topmost=1500000, count_path=3)
    words = str(e.value).split()
    need, have = int(words[words.index("needs") + 1]), int(words[words.index("its") + 1])
    records = int(words[words.index("lists") + 1])

    def lists(cap):
        return -(-16 * cap // 256) * 256 + 2 * (-(-32 * cap // 256) * 256)

    cap = records
    while need - lists(records) + lists(cap) > have:
        cap -= 1
    k = 1500000 - (records - cap)
    with ge.Panel.from_planes(bits, valid, n) as h:
        got, _ = h.scan_noalloc(m0, m1, topmost=k, count_path=3)
        assert len(got) == k
        assert_same(got, h.scan(m0, m1, topmost=k, count_path=3)[0], "longest")
        with pytest.raises(ge.GepiError):
            h.scan_noalloc(m0, m1, topmost=k + 16, count_path=3)
