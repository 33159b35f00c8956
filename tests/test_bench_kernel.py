"""What the benchmark names and prices as a scan's count kernel."""
import bench


def test_products_of_a_variant_pair():
    assert bench.count_kernel(3, False) == ("k_count_f4g", 9)
    assert bench.count_kernel(3, True) == ("k_count_f4c", 4)
    assert [bench.count_kernel(p, c) for p in (4, 2, 1) for c in (False, True)] == [
        ("k_count_f4", 9)] * 2 + [("k_count_mfma", 9)] * 2 + [("k_count_popc", 9)] * 2


def test_compute_type_by_path():
    assert bench.DTYPES[3] == bench.DTYPES[4] and bench.DTYPES[4].startswith("fp4")
    assert bench.DTYPES[2] == "i8" and 1 not in bench.DTYPES
