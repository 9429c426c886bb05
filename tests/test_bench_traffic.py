"""The traffic summaries that bench.py reports beside its times (profiles/*_hbm_traffic.json): they are of the kernels that
the library holds, and a kernel's bytes are those of one launch."""
import json
import os
import re
import subprocess

import pytest

import bench
from fortrancfd_amd.build import LIB

WORKLOADS = sorted(bench.TRAFFIC_PROFILES)


def summary(workload):
    return json.load(open(os.path.join(bench.REPO, "profiles", bench.TRAFFIC_PROFILES[workload])))["kernels"]


@pytest.mark.parametrize("workload", WORKLOADS)
def test_kernels_are_the_library_s(workload):
    stubs = set(re.findall(r"__device_stub__(\w+(?:<[^>]*>)?)\(", subprocess.run(["nm", "-C", LIB], check=True,
                                                                                capture_output=True, text=True).stdout))
    assert stubs
    kernels = [re.search(r"(\w+(?:<[^>]*>)?)\(", k.replace("(anonymous namespace)::", "")).group(1)
               for k in summary(workload) if "fcfd::" in k]
    assert kernels and not set(kernels) - stubs


@pytest.mark.parametrize("workload", WORKLOADS)
@pytest.mark.parametrize("kernel", ["k_flux", "k_stage_end", "k_wave_speed", "k_chem_screen"])
def test_bytes_of_one_launch(workload, kernel):
    got, src = bench.measured_traffic(workload, kernel)
    each = [r["read_bytes"] + r["write_bytes"] for name, r in summary(workload).items() if kernel + "<" in name]
    assert (got is None) == (not each)
    if each:
        assert min(each) <= got <= max(each) and src.startswith("profiles")
