"""Accuracy of the binary64 row transforms, on the host: the register DFTs and
twiddles of hy_fft.hpp against a long-double DFT.

The bound is the RMS error of the plain transform of the same row: radix 3, 8, 4
and 2 stages with one correctly rounded table factor per element between them,
measured by the same program (1.13e-16 at 6 to 2.20e-16 at 1024 elements), with 2% for
the sampling of the rows.  Factors that are not correctly rounded, or roundings that
the plain transform does not have, exceed it (2.2 to 2.5e-16 at 192, 384 and 1024)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PLAIN = {6: 1.129e-16, 12: 1.232e-16, 24: 1.419e-16, 48: 1.595e-16, 96: 1.726e-16, 192: 1.882e-16, 384: 2.010e-16,
         8: 1.016e-16, 16: 1.226e-16, 32: 1.377e-16, 64: 1.592e-16, 128: 1.776e-16, 256: 1.881e-16,
         512: 2.072e-16, 1024: 2.200e-16}


@pytest.fixture(scope="module")
def errors(tmp_path_factory):
    from hyowon_amd import build
    exe = str(tmp_path_factory.mktemp("fft_rows") / "fft_rows")
    subprocess.run([build.hipcc(), "-x", "hip", "--offload-host-only", "-O1", "-std=c++20", "-ffp-contract=off",
                    f"-I{build.CSRC}", os.path.join(ROOT, "tests", "cpp", "fft_rows.hip"), "-o", exe], check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout
    return {int(f[0]): [float(v) for v in f[1:]] for f in (line.split() for line in out.splitlines())}


@pytest.mark.parametrize("length", sorted(PLAIN))
def test_row_transform_error(errors, length):
    for name, err in zip(("forward", "inverse", "x inverse"), errors[length]):
        assert err <= 1.02 * PLAIN[length], (name, err)
