"""The traffic that bench.py reports is looked up by kernel name in the committed counter summaries: the names have to be those of
the kernels that the profiled build launches, or the figure silently becomes null."""
import os

import pytest

import bench

PROFILES = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "profiles")


@pytest.mark.parametrize("workload,mode", [("limited_2p7b", "keep"), ("limited_2p7b", "recompute"), ("irregular", "keep"), ("large_vocab", "keep"), ("tiny_track", "keep")])
def test_traffic_of_every_large_kernel_is_found(workload, mode):
    for kind in bench.PROFILE_KERNEL:
        if kind != "recompute" or mode == "recompute":
            assert bench.measured_traffic(workload, mode, kind), (workload, mode, kind)


def test_traffic_of_an_unknown_workload_is_none():
    assert bench.measured_traffic("none_such", "keep", "dw") is None


def test_profiles_name_kernels_of_this_source():
    src = "".join(open(os.path.join(os.path.dirname(PROFILES), "slowrun_amd", "csrc", f)).read()
                  for f in sorted(os.listdir(os.path.join(os.path.dirname(PROFILES), "slowrun_amd", "csrc"))) if f.endswith((".h", ".hip")))
    for f in sorted(os.listdir(PROFILES)):
        if f.startswith(("bench_", "cases_", "kernel_resources")):
            for ln in open(os.path.join(PROFILES, f)):
                for word in ln.split():
                    name = word.split("<")[0]
                    if name.endswith("_kernel") and name.startswith(("fwd_", "bwd_", "quantize_", "prep_", "amax_")):
                        assert name in src, f"{f} names {name}, which the library does not have"
