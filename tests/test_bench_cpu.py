"""The benchmark's use of recorded profiles: a count is taken only for the lists and the
kernel sources that it was measured with."""
import json

import bench


def test_profiles_hold_for_their_kernels_only(tmp_path):
    path = str(tmp_path / "p.json")
    good = {"sources": bench.kernel_sources(), "pairs": 12, "fp32_flops_per_launch": 3.0}
    with open(path, "w") as f:
        json.dump({"a": good, "b": dict(good, sources="0" * 16), "c": {"fp32_flops_per_launch": 3.0}}, f)
    assert bench.profiled(path, "a", 12) == good
    assert bench.profiled(path, "a", 13) is None  # other lists
    for key in "bcd":  # other kernels, an unmarked record, none
        assert bench.profiled(path, key, 12) is None
    assert bench.profiled(str(tmp_path / "none.json"), "a", 12) is None
