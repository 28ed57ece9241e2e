"""Sizes of launches (micm_amd/csrc/launch_rules.hpp) over the ranges they are asked for."""
import ctypes
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOLVER = os.path.join(ROOT, "micm_amd", "csrc", "solver.hip")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("rules") / "librules.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", os.path.join(ROOT, "tests", "launch_rules_harness.cpp"),
                    "-o", out], check=True)
    lib = ctypes.CDLL(out)
    lib.tile_cells_host.argtypes = [ctypes.c_int64, ctypes.c_int64]
    lib.with_block_host.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int64, ctypes.c_int]
    lib.slices_host.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.POINTER(ctypes.c_int64), ctypes.c_int64]
    lib.staging_bytes_host.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int64]
    lib.staging_bytes_host.restype = ctypes.c_int64
    lib.slices_host.restype = ctypes.c_int64
    return lib


@pytest.mark.parametrize("kernel", ["k_lu_decompose_tiled", "k_lu_solve_tiled"])
@pytest.mark.parametrize("limit", [64 * 1024 - 64, 160 * 1024 - 64])
def test_a_tile_has_a_kernel_of_its_size(lib, kernel, limit):
    """The grid is sized for the tile that the rule gives, so the launch needs a kernel built for
    exactly that tile: with a smaller one, cells past its first would be left out."""
    built = {int(tc) for tc in re.findall(rf"LAUNCH_TILED\({kernel}<(\d+)>", open(SOLVER).read())}
    for doubles in range(1, 22000):
        tc = lib.tile_cells_host(doubles, limit)
        assert tc == 0 or tc in built, (doubles, tc)
        assert (tc == 0) == (doubles * 8 > limit), (doubles, tc)
        assert tc <= 1 or 2 * doubles * tc * 8 <= limit, (doubles, tc)


@pytest.mark.parametrize("cells,threads", [
    (c, t) for c in (0, 1, 64, 513, 1 << 22, (1 << 28) + 37, (1 << 32) + 1)
    for t in (1, 3, 16, 20, 210, 256, 511, 1 << 20) if c * t <= 1 << 40])
def test_slices_cover_the_cells_and_fit_a_launch(lib, cells, threads):
    """Each cell is in one slice, slices start at whole groups for every XCD, and a slice's threads,
    rounded up to such groups, are fewer than the 2^32 that a launch takes."""
    most = 4096
    out = (ctypes.c_int64 * (2 * most))()
    n = lib.slices_host(cells, threads, out, most)
    assert n >= 0
    at = 0
    for q in range(n):
        first, count = out[2 * q], out[2 * q + 1]
        assert first == at and count > 0 and first % 512 == 0
        assert (count + 511) // 512 * 512 * threads < 1 << 32
        at += count
    assert at == cells
    if cells * threads <= 1 << 30:
        assert n == min(cells, 1)  # ordinary calls stay one launch


@pytest.mark.parametrize("species,reactions", [(1, 0), (3, 2), (9, 70), (20, 50), (60, 200), (210, 560), (5000, 1)])
def test_pinned_memory_of_a_state_is_what_a_copy_of_it_uses(lib, species, reactions):
    """No pinned byte that no copy to the host reaches; pinned memory for results up to 256 KiB and
    for grouped arrays below 16."""
    for cells in (1, 2, 63, 64, 65, 400, 1000, 3855, 3856, 4096, 10000, 100000, 1 << 28):
        padded = (cells + 63) // 64 * 64
        copies = [68 * cells, 8 * padded * species, 8 * padded * reactions]
        got = lib.staging_bytes_host(cells, species, reactions)
        used = [c for c, most in zip(copies, (256 * 1024, 16 * 1024 - 1, 16 * 1024 - 1)) if c <= most]
        assert got == max(used, default=0)


@pytest.mark.parametrize("factor,products,cells,lu,substitution", [
    (131, 200, 768, True, True), (131, 200, 769, False, False), (1100, 9000, 5000, False, False),
    (1304, 7668, 769, True, True), (2381, 6986, 20000, True, True), (8548, 121036, 4096, True, True),
    (1252, 1882, 769, False, False), (1252, 1882, 100000, False, False), (1417, 4291, 8000, False, True),
    (1697, 3653, 2048, False, True), (1697, 3653, 2049, True, True), (1700, 2000, 4000, True, False)])
def test_dense_block_by_entries_products_and_cells(lib, factor, products, cells, lu, substitution):
    assert bool(lib.with_block_host(factor, products, cells, 0)) == lu
    assert bool(lib.with_block_host(factor, products, cells, 1)) == substitution
