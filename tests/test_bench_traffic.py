"""The roofline record's counter bytes are those of the kernel that it names."""
import json

import bench


def test_another_kernels_counters_are_not_used(tmp_path):
    f = tmp_path / "traffic.json"
    f.write_text(json.dumps({"op": {"traffic_bytes_per_launch": 5.0, "kernel": "k_old"}}))
    assert bench.counter_traffic("op", "k_old", f) == 5.0
    assert bench.counter_traffic("op", bench.ROOF_KERNEL, f) is None
    assert bench.counter_traffic("other", "k_old", f) is None
    assert bench.counter_traffic("op", "k_old", tmp_path / "missing.json") is None


def test_the_recorded_kernel_is_the_one_that_runs(nbx):
    assert bench.counter_traffic("axhelm_bk_f64_n7_32cube", bench.ROOF_KERNEL)
    mangled = b"_ZN3nbx8k_axhelmIdLi8ELi1ELb1ELb0EdE"  # ROOF_KERNEL in the library
    from pathlib import Path
    assert mangled in (Path(nbx.__file__).parent / "libnbx.so").read_bytes()
