"""The factor's dense block (micm_amd/csrc/tail.hpp): its tables executed on the CPU give the
oracle's factors and solutions bit for bit, with the block's structural zeros multiplied
through (finite values) and with every product tested against the fill pattern."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from helpers import bits_equal
from mechanisms import all_rate_types, ts1_inputs, ts1_mechanism
from micm_amd import synthetic
from oracle import Oracle

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_dp = ctypes.POINTER(ctypes.c_double)


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("tail") / "libtail_harness.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-ffp-contract=off",
                    os.path.join(ROOT, "tests", "tail_harness.cpp"),
                    os.path.join(ROOT, "micm_amd", "csrc", "mechanism.cpp"), "-o", out], check=True)
    lib = ctypes.CDLL(out)
    lib.tail_factor_solve.argtypes = [ctypes.c_void_p, _dp, ctypes.c_double, ctypes.c_int32, _dp, _dp, _dp]
    lib.tail_shape.argtypes = [ctypes.c_void_p, ctypes.POINTER(ctypes.c_int64)]
    return lib


# (mechanism, inputs, whether it has a block: at least sixteen species)
CASES = {
    "readme": (synthetic.readme_mechanism, lambda d, n: synthetic.readme_inputs(n), False),
    "all_types": (all_rate_types, None, False),
    "16_30": (lambda: synthetic.random_mechanism(16, 30, {0: 30}, 5), synthetic.inputs_60_200, True),
    "17_40": (lambda: synthetic.random_mechanism(17, 40, {0: 40}, 6), synthetic.inputs_60_200, True),
    "20_50": (synthetic.mechanism_20_50, synthetic.inputs_60_200, True),
    "60_200": (synthetic.mechanism_60_200, synthetic.inputs_60_200, True),
    "210_560": (synthetic.mechanism_210_560, synthetic.inputs_210_560, True),
    "210_560_literal": (lambda: synthetic.mechanism_210_560(products_from="all"), synthetic.inputs_210_560, True),
    "ts1": (ts1_mechanism, ts1_inputs, True),
}


@pytest.mark.parametrize("name", list(CASES))
def test_block_tables_reproduce_doolittle(harness, name):
    make, inputs, has_block = CASES[name]
    desc = make()
    cdesc = ctypes.byref(desc.as_c())
    o = Oracle(desc, 4)
    if inputs is None:
        rng = np.random.default_rng(7)
        y, cond = rng.uniform(1e-6, 1.0, (1, desc.n_species)), np.array([[280.0, 9e4, 38.0]])
        custom = rng.uniform(1e-6, 1e-2, (1, o.n_custom))
    else:
        cells = inputs(desc, 1)
        y, cond, custom = cells.variables[:, o.species_order()], cells.conditions, cells.custom
    k = o.rate_constants(cond, custom)
    jac, f = o.jacobian(k, y), o.forcing(k, y)
    alpha = 1.0 / (300.0 * 0.57282)
    _, lo_ref, up_ref = o.lu(jac, alpha)
    x_ref = o.lu_solve(lo_ref, up_ref, f)
    for masked in (0, 1):
        lo, up, x = np.zeros(lo_ref.shape[1]), np.zeros(up_ref.shape[1]), f[0].copy()
        size = harness.tail_factor_solve(cdesc, np.ascontiguousarray(jac[0]).ctypes.data_as(_dp), alpha, masked,
                                         lo.ctypes.data_as(_dp), up.ctypes.data_as(_dp), x.ctypes.data_as(_dp))
        assert (size > 0) == has_block and size >= 0
        if size:
            assert size % 16 == 0 and size <= min(64, desc.n_species)
            assert bits_equal(lo, lo_ref[0]) and bits_equal(up, up_ref[0])
            assert bits_equal(x, x_ref[0])
