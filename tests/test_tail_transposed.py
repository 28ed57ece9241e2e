"""The transposed substitutions with the factor's dense block: the block's tables executed on the
CPU give the solution of a row by row substitution bit for bit."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from helpers import bits_equal
from mechanisms import ts1_mechanism
from micm_amd import synthetic

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_dp = ctypes.POINTER(ctypes.c_double)


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("tail_transposed") / "libtail_transposed_harness.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-ffp-contract=off",
                    os.path.join(ROOT, "tests", "tail_transposed_harness.cpp"),
                    os.path.join(ROOT, "micm_amd", "csrc", "mechanism.cpp"), "-o", out], check=True)
    lib = ctypes.CDLL(out)
    lib.tail_transposed.argtypes = [ctypes.c_void_p, _dp, ctypes.c_int64, _dp, _dp, _dp]
    return lib


def _random(n_species, n_reactions):
    return lambda: synthetic.random_mechanism(n_species, n_reactions, {0: n_reactions}, 100 + n_species)


CASES = {
    "readme": synthetic.readme_mechanism,
    "16_30": _random(16, 30),
    "17_40": _random(17, 40),
    "20_50": synthetic.mechanism_20_50,
    "60_200": synthetic.mechanism_60_200,
    "65_180": _random(65, 180),
    "210_560": synthetic.mechanism_210_560,
    "210_560_literal": lambda: synthetic.mechanism_210_560(products_from="all"),
    "256_700": _random(256, 700),
    "ts1": ts1_mechanism,
}


@pytest.mark.parametrize("name", list(CASES))
def test_transposed_tables(harness, name):
    desc = CASES[name]()
    n, capacity = desc.n_species, desc.n_species ** 2
    rng = np.random.default_rng(n)
    # quotients and products stay near one, so that no value reaches a limit of the format
    alu, b = rng.uniform(0.5, 1.5, capacity) * rng.choice([-0.2, 0.2], capacity), rng.standard_normal(n)
    x, ref = np.zeros(n), np.zeros(n)
    size = harness.tail_transposed(ctypes.byref(desc.as_c()), alu.ctypes.data_as(_dp), capacity, b.ctypes.data_as(_dp),
                                   x.ctypes.data_as(_dp), ref.ctypes.data_as(_dp))
    assert size == 0 if n < 16 else (size > 0 and size % 16 == 0)
    if size:
        keep = np.isfinite(ref)
        assert keep.any() and bits_equal(x[keep], ref[keep]) and np.array_equal(np.isfinite(x), keep)
