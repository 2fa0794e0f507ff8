"""The reciprocals of the thermal strips (geoflac_amd/csrc/gf_rcp.h): the header itself compiled
for the host against IEEE division, with its guard; and the device's, from the hardware's
estimate, against the host's division, bit for bit."""
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def test_header_reciprocals_are_correctly_rounded(tmp_path):
    exe = str(tmp_path / "rcp_header_check")
    try:
        subprocess.run(["g++", "-O2", "-mfma", "-ffp-contract=off", "-std=c++17",
                        "-I", os.path.join(HERE, "..", "geoflac_amd", "csrc"),
                        os.path.join(HERE, "csrc", "rcp_header_check.cpp"), "-o", exe, "-lm"],
                       check=True, capture_output=True, text=True)
    except OSError as e:  # no C++ compiler
        pytest.skip("g++ unavailable: %s" % e)
    out = subprocess.run([exe, "10000000"], check=True, capture_output=True, text=True).stdout
    assert [int(v) for v in out.split()] == [0, 0, 0]


def _operands(n):
    rng = np.random.default_rng(5)
    ones = np.uint64((1 << 52) - 1)
    m = rng.integers(0, 1 << 52, n, dtype=np.uint64)
    m[::16] = ones - rng.integers(0, 4, m[::16].size, dtype=np.uint64)
    m[1::16] = rng.integers(0, 4, m[1::16].size, dtype=np.uint64)
    e = rng.integers(-420, 421, n).astype(np.int64)
    e[3::8] = rng.integers(-1022, 1023, e[3::8].size)  # (beyond the guard: the device divides)
    u = ((e + 1023).astype(np.uint64) << np.uint64(52)) | m | (rng.integers(0, 2, n, dtype=np.uint64) << np.uint64(63))
    return u.view(np.float64)


@pytest.mark.gpu
def test_device_reciprocals_equal_division():
    from geoflac_amd import gpu
    x = _operands(1 << 22)
    print("case: %d reciprocals" % x.size, flush=True)
    with np.errstate(all="ignore"):
        q = 1.0 / x
        back = 1.0 / q
    assert np.array_equal(gpu.math_check(4, x).view(np.uint64), q.view(np.uint64))
    assert np.array_equal(gpu.math_check(5, x).view(np.uint64), back.view(np.uint64))
