"""The autotuner on a mechanism that says which kernel a shape launches
(micm_hip_mechanism_cooperative_kernel): shapes that are one launch are timed once, the LU blockings
only where the kernel has the LU schedule, and the near tie of the two register budgets holds
whatever label the wider build is kept under."""
import types

import numpy as np
import pytest

from micm_amd import _lib, autotune

LEVELS, COMPACT, BLOCK, LANE = _lib.KERNEL_LEVELS, _lib.KERNEL_COMPACT, _lib.KERNEL_BLOCK, _lib.KERNEL_LANE


def block_kernels(default_waves):
    """16 to 256 species."""
    def kernel(stages, threads, stage, n_cells=1):
        if stage < 0 and threads in (0, 256) or threads == 256 and stage >= 4:
            return BLOCK, 256, 0, {5: 3, 6: 2, 7: 2}.get(stage, default_waves)
        return (COMPACT if stage < 0 else LEVELS), threads, max(stage, 0) & 3, 0
    return kernel


def lane_kernels(stages, threads, stage, n_cells=1):
    """The smallest mechanisms."""
    if stage < 0:
        return LANE, 0, 0, 0
    return (COMPACT, threads, 0, 0) if threads == 256 and stage >= 4 else (LEVELS, threads, stage & 3, 0)


def tune(monkeypatch, kernel, seconds, tag):
    """autotune with times by kernel; (choice, [(label, cells, blocking)])."""
    calls = []

    def fake(mech, y, k, dt, params, candidates, repeats, verbose, give_up=None, lu_blocking=0):
        out = {}
        for c in candidates:
            calls.append((c[0], y.shape[0], lu_blocking))
            what = kernel(4, c[3], c[4]) if c[1] == _lib.SOLVE_COOPERATIVE else (c[0],)
            # every run a little faster than the last: noise that must not pick a blocking
            out[c[0]] = seconds(what) * (1e-3 + 1e-6 * y.shape[0]) * (0.95 if lu_blocking else 1.0)
        return out

    monkeypatch.setattr(autotune, "_time_candidates", fake)
    mech = types.SimpleNamespace(
        info=types.SimpleNamespace(n_species=tag, n_reactions=1, nnz_jacobian=1, nnz_lower=1, nnz_upper=1,
                                   lu_multiply_adds=1),
        cooperative_supported=lambda stages: True, cooperative_kernel=kernel)
    state = types.SimpleNamespace(n_cells=100000, get_variables=lambda: np.zeros((100000, 1)),
                                  get_rate_constants=lambda: np.zeros((100000, 1)))
    return autotune.autotune(mech, state, 30.0, types.SimpleNamespace(stages=4)), calls


@pytest.fixture(autouse=True)
def _fresh_cache():
    autotune._cache.clear()
    yield
    autotune._cache.clear()


@pytest.mark.parametrize("kernel", [block_kernels(2), block_kernels(3), lane_kernels])
def test_each_kernel_is_timed_once_and_without_blockings(monkeypatch, kernel):
    best = BLOCK if kernel is not lane_kernels else LANE
    choice, calls = tune(monkeypatch, kernel, lambda k: 1.0 if k[0] == best else 1.9, tag=900)
    shapes = {c[0]: c for c in autotune.CANDIDATES}
    pilot = [shapes[label] for label, n, b in calls if n == 256]
    kernels = [kernel(4, c[3], c[4]) for c in pilot if c[1] == _lib.SOLVE_COOPERATIVE]
    assert len(kernels) == len(set(kernels))
    # nothing is left out
    assert set(kernels) == {kernel(4, c[3], c[4]) for c in autotune.CANDIDATES if c[1] == _lib.SOLVE_COOPERATIVE}
    assert {c[0] for c in pilot if c[1] != _lib.SOLVE_COOPERATIVE} >= {"persistent+handoff16", "plain"}
    assert all(b == 0 for _, _, b in calls)
    assert choice["lu_blocking"] == 0 and choice["lu_blocking_seconds"] == {}
    assert kernel(4, choice["threads"], choice["stage"])[0] == best


def test_blockings_are_timed_where_the_kernel_has_the_schedule(monkeypatch):
    choice, calls = tune(monkeypatch, block_kernels(2), lambda k: 1.0 if k == (COMPACT, 128, 0, 0) else 1.5, tag=901)
    assert choice["label"] == "cooperative128" and choice["lu_blocking"] in autotune.LU_BLOCKINGS
    assert {b for label, n, b in calls if label == "cooperative128"} == {0, *autotune.LU_BLOCKINGS}


@pytest.mark.parametrize("default_waves", [2, 3])
@pytest.mark.parametrize("margin,waves", [(0.995, 2), (0.98, 3)])
def test_near_tie_of_the_register_budgets(monkeypatch, margin, waves, default_waves):
    seconds = {(BLOCK, 256, 0, 2): 1.0, (BLOCK, 256, 0, 3): margin}
    choice, _ = tune(monkeypatch, block_kernels(default_waves), lambda k: seconds.get(k, 1.9), tag=902)
    assert block_kernels(default_waves)(4, choice["threads"], choice["stage"])[3] == waves
