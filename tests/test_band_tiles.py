"""The band kernels' tile rule on the CPU: every tile's union fits the 32 slots
that a staged row has."""
import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BUILD = os.path.join(ROOT, "tests", "native", "_build")


@pytest.fixture(scope="module")
def host_band():
    os.makedirs(BUILD, exist_ok=True)
    out = os.path.join(BUILD, "libband_host.so")
    subprocess.run(["/opt/rocm/bin/hipcc", "-O1", "-std=c++17", "-fPIC", "-shared",
                    "-I" + os.path.join(ROOT, "natten-mps_amd", "csrc"), "-I" + os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "native", "band_host.cpp"), "-o", out], check=True)
    return ctypes.CDLL(out)


@pytest.mark.parametrize("kernel", range(2, 17))
def test_unions_fit_a_staged_row(host_band, kernel):
    for key in (0, 1):
        cols = 1 << host_band.host_band_columns(kernel, key)
        assert cols in (8, 16)
        for d in (1, 2, 3, 5):
            for causal in (0, 1):
                # past 6 kernels per class the borders no longer meet
                assert host_band.host_widest_union(6 * kernel * d + 40, kernel, d, causal, cols, key) <= 32


def test_wider_kernels_are_declined_on_the_key_side(host_band):
    assert host_band.host_band_columns(17, 1) == -1 and host_band.host_band_columns(18, 0) == -1
