"""CPU check, bit for bit: the superbee limiter as medians against the reference's expression
(cpu_slope_limiters.hpp:30-54)."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "limiter_host_check.hip")
OUT = os.path.join(HERE, "_build", "liblimiter_host_check.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    os.makedirs(os.path.dirname(OUT), exist_ok=True)
    deps = [SRC] + [os.path.join(HERE, "..", "vlasiator_amd", "csrc", f) for f in ("vacc_recon.h", "vacc_common.h")]
    if not os.path.exists(OUT) or os.path.getmtime(OUT) < max(os.path.getmtime(d) for d in deps):
        subprocess.run([HIPCC, "--offload-arch=gfx950", "-O2", "-std=c++17", "-fPIC", "-shared",
                        "-ffp-contract=off", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                        SRC, "-o", OUT], check=True, capture_output=True)
    return C.CDLL(OUT)


def _ptr(a):
    return a.ctypes.data_as(C.c_void_p)


def _reference_superbee(a, b):
    f = np.float32
    def pick(s1, s2, smaller):
        first = np.abs(s1) < np.abs(s2) if smaller else np.abs(s1) > np.abs(s2)
        return np.where((s1 * s2).astype(f) <= 0, f(0), np.where(first, s1, s2)).astype(f)
    return pick(pick(a, (f(2) * b).astype(f), True), pick((f(2) * a).astype(f), b, True), False)


def test_superbee_bits(lib):
    """Signs, ties, twofold ratios, zeros of either sign, and magnitudes down to subnormals, where
    the reference's product tests underflow."""
    rng = np.random.default_rng(1)
    n = 400_000
    a = (rng.choice([-1.0, 1.0], n) * 10.0 ** rng.uniform(-45, 30, n)).astype(np.float32)
    ratio = rng.choice([1.0, 2.0, 0.5, 0.0, -1.0, 1e-20, 1e20], n) * np.where(rng.random(n) < 0.5, 1.0, 10.0 ** rng.uniform(-3, 3, n))
    with np.errstate(all="ignore"):
        b = (a * ratio).astype(np.float32)
        b[~np.isfinite(b)] = np.float32(1.0)
        a[rng.random(n) < 0.01] = np.float32(-0.0)
        want = _reference_superbee(a, b)
    got = np.zeros(n, np.float32)
    lib.superbee_batch(_ptr(a), _ptr(b), n, _ptr(got))
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
