"""The workgroup's running sum (micm_amd/csrc/ordered_sum.hpp) executed on the host with every
thread of the workgroup, at both of its sizes and with the wavefronts in either order between
barriers: the result is that of adding one term after another, bit for bit, on every thread, and
all wavefronts meet at the same barriers.  Inputs reach each branch: whole tiles of zeros before
the first other term, sums that are outside the range of the parallel form when the tiles start,
ties, new binades, overflow and NaN."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("sum") / "libsum_workgroup.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-ffp-contract=off", "-Wno-unknown-pragmas",
                    os.path.join(ROOT, "tests", "ordered_sum_workgroup.cpp"), "-o", out], check=True)
    lib = ctypes.CDLL(out)
    lib.ordered_sum_workgroup.argtypes = [ctypes.POINTER(ctypes.c_double), ctypes.c_int64, ctypes.c_int, ctypes.c_int,
                                          ctypes.POINTER(ctypes.c_double)]
    return lib


CHAIN, TILE = 2048, 8192


def sums():
    r = np.random.default_rng(11)
    some = lambda n: r.uniform(0.0, 1.0, n)
    out = {
        "squares": r.standard_normal(20011) ** 2,
        "wide": np.exp(r.uniform(-80, 20, 20000)) ** 2,
        "ties": np.concatenate([[4.0], r.integers(0, 16, 20000) * 2.0 ** -52]),
        "all_zero": np.zeros(CHAIN + 2 * TILE + 5),
        # the first term that is not zero in a tile of its own, by the wavefront that reaches it
        "zero_tile_first_wave": np.concatenate([np.zeros(CHAIN + TILE), some(700)]),
        "zero_tile_last_wave": np.concatenate([np.zeros(CHAIN + 2 * TILE - 40), some(700)]),
        "zero_tiles": np.concatenate([np.zeros(CHAIN + 2 * TILE + 3000), some(9000)]),
        # the chain ends below the parallel form's range, and the first wavefront takes it in
        "small_chain": np.concatenate([np.full(CHAIN, 1e-290), some(9000)]),
        "small_tiles": np.concatenate([np.full(CHAIN + TILE + 77, 1e-290), some(3000)]),
        "large": np.concatenate([np.full(CHAIN, 1e280), r.uniform(0, 1e300, 9000)]),
        "overflow": np.concatenate([some(CHAIN + 300), [1e308, 1e308], some(9000)]),
        "nan": np.concatenate([some(CHAIN + 300), [np.nan], some(9000)]),
    }
    return out


SUMS = sums()


@pytest.mark.parametrize("order", ["ascending", "descending"])
@pytest.mark.parametrize("threads", [1024, 512])
@pytest.mark.parametrize("name", list(SUMS))
def test_workgroup_sum_is_the_sequential_sum(lib, name, threads, order):
    t = np.ascontiguousarray(SUMS[name])
    acc = 0.0
    with np.errstate(all="ignore"):
        for v in t.tolist():
            acc += v
    got = ctypes.c_double()
    status = lib.ordered_sum_workgroup(t.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), len(t), threads,
                                       order == "descending", ctypes.byref(got))
    assert status != 1, "wavefronts wait at different barriers"
    assert status == 0, "threads end with different sums"
    got = got.value
    assert np.array([got]).view(np.int64) == np.array([acc]).view(np.int64) or (np.isnan(got) and np.isnan(acc))
