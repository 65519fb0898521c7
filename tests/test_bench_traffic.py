"""bench.py's measured HBM traffic comes from the committed counter summary of exactly the
kernel that a stage runs: every stage kernel of the default workload is a kernel of
the built library, the summary's kernels still exist, and an instantiation that the
summary does not hold is reported as missing."""
import json
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROFILE = os.path.join(ROOT, "profiles", "pm_kdk_step_512p_1024m_fp32_traffic.json")
PLAN = {"variant": {"z_r2c": 2, "y_fwd": 2, "x_green": 3, "y_bwd": 2, "z_c2r": 1}}


@pytest.fixture(scope="module")
def library_kernels():
    from hyowon_amd import build
    if not os.path.exists(build.LIB):
        build.build()
    out = subprocess.run(["nm", "-C", build.LIB], check=True, capture_output=True, text=True).stdout
    return {re.sub(r"^void ", "", n).split("(")[0].replace("__device_stub__", "")
            for n in re.findall(r"\b(?:void )?hy::__device_stub__.*", out)}


def _name(kernel):
    return re.sub(r"^void ", "", kernel).split("(")[0]


def test_summary_kernels_exist(library_kernels):
    with open(PROFILE) as f:
        kernels = json.load(f)["kernels"]
    gone = [k for k in kernels if "hy::" in k and _name(k) not in library_kernels]
    assert not gone, gone


@pytest.mark.parametrize("stage", ["deposit", "fft_z_r2c", "fft_y_fwd", "fft_x_green", "fft_y_bwd", "fft_z_c2r",
                                   "gather_kdk"])
def test_stage_has_its_own_kernel(stage):
    import bench
    bytes_, source = bench.measured_traffic(stage, 512, 1024, "fp32", PLAN)
    assert source == "profiles/pm_kdk_step_512p_1024m_fp32_traffic.json"
    assert 6e9 < bytes_ < 2e10


def test_another_instantiation_is_missing(monkeypatch):
    import bench
    other = {"variant": dict(PLAN["variant"], x_green=0)}
    assert bench.measured_traffic("fft_x_green", 512, 1024, "fp32", other)[0] is None
    monkeypatch.setitem(bench.STAGE_KERNEL, "gather_kdk", "void hy::k_gather_kdk<float, float, true, true, false")
    assert bench.measured_traffic("gather_kdk", 512, 1024, "fp32", PLAN)[0] is None
