"""A running sum formed in parallel (micm_amd/csrc/ordered_sum.hpp): its arithmetic on the host
against adding one term after another, bit for bit, on sums that tie, cross binades, start from
zeros and leave the double range."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("sum") / "libsum_harness.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-ffp-contract=off",
                    os.path.join(ROOT, "tests", "ordered_sum_harness.cpp"), "-o", out], check=True)
    lib = ctypes.CDLL(out)
    lib.ordered_sum_host.restype = ctypes.c_double
    lib.ordered_sum_host.argtypes = [ctypes.POINTER(ctypes.c_double), ctypes.c_int64]
    return lib


def sums():
    """name -> terms; the last ones tie often (few bits, all multiples of half a unit)."""
    r = np.random.default_rng(3)
    out = {
        "squares": r.standard_normal(20000) ** 2,
        "wide": np.exp(r.uniform(-80, 20, 20000)) ** 2,
        "tiny_then_large": np.concatenate([np.exp(r.uniform(-300, -200, 500)), r.uniform(0, 1, 3000)]),
        "zeros": np.concatenate([np.zeros(1000), r.uniform(0, 1, 77), np.zeros(100)]),
        "all_zero": np.zeros(50),
        "one": np.array([0.1]),
        "denormal": np.full(300, 5e-324),
        "huge": np.concatenate([r.uniform(0, 1e300, 100), [1e308, 1e308, 1e308], r.uniform(0, 1, 40)]),
        "infinite": np.concatenate([r.uniform(0, 1, 100), [np.inf], r.uniform(0, 1, 100)]),
        "nan": np.concatenate([r.uniform(0, 1, 100), [np.nan], r.uniform(0, 1, 100)]),
        "ulp_ties": np.concatenate([[1.0], np.full(5000, 2.0 ** -53), np.full(5000, 3 * 2.0 ** -53)]),
        "half_ties": np.concatenate([[4.0], r.integers(0, 16, 20000) * 2.0 ** -52]),
        "coarse": np.concatenate([[2.0 ** 52], r.integers(0, 9, 20000) * 0.5]),
    }
    return out


@pytest.mark.parametrize("name", list(sums()))
def test_parallel_sum_is_the_sequential_sum(lib, name):
    t = np.ascontiguousarray(sums()[name])
    acc = 0.0
    with np.errstate(all="ignore"):
        for v in t.tolist():
            acc += v
    got = lib.ordered_sum_host(t.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), len(t))
    assert np.array([got]).view(np.int64) == np.array([acc]).view(np.int64) or (np.isnan(got) and np.isnan(acc))
