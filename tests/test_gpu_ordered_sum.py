"""micm_hip_normalized_error_state where its running sum is formed in parallel: States of more
terms than the leading chain, up to several tiles and a partial one, in Matrix and VectorMatrix
order, against the reference's arithmetic bit for bit; errors that tie (few bits), that start
with zeros, and that overflow."""
import numpy as np
import pytest

from helpers import dev
from micm_amd import _lib, synthetic
from oracle import OraclePortableMath

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["random", "ties", "zeros", "wide", "overflow"])
@pytest.mark.parametrize("n_cells,group", [(103, 1), (511, 4), (1200, 1), (1201, 64)])
def test_state_error_of_large_states(n_cells, group, kind):
    print(f"state error: {n_cells} cells, group {group}, {kind}", flush=True)
    import torch
    desc = synthetic.mechanism_20_50()
    mech, oracle = _lib.Mechanism(desc), OraclePortableMath(desc, 4)
    n = mech.n_species
    r = np.random.default_rng(n_cells)
    y, ynew = r.uniform(0.0, 1e-3, (2, n_cells, n))
    atol = np.full(n, 1e-3)
    rtol = 1e-6
    err = r.standard_normal((n_cells, n)) * 1e-3
    if kind == "ties":
        y, ynew, rtol = np.zeros_like(y), np.zeros_like(y), 0.0
        atol = np.full(n, 2.0 ** -10)
        err = r.integers(0, 4, (n_cells, n)) * 2.0 ** -10 * np.where(r.random((n_cells, n)) < 0.5, 1.0, 2.0 ** -26)
    elif kind == "zeros":
        err[: n_cells // 2] = 0.0
    elif kind == "wide":
        err *= np.exp(r.uniform(-60.0, 40.0, err.shape))
    elif kind == "overflow":
        err[n_cells - 2] = 1e200
    out = torch.zeros(1, dtype=torch.float64, device="cuda")
    bufs = [dev(a) for a in (y, ynew, err)]
    a = torch.from_numpy(atol).cuda()
    mech.normalized_error_state(n_cells, *(b.data_ptr() for b in bufs), a.data_ptr(), rtol, group, out.data_ptr())
    got = float(out.cpu()[0])
    want = float(oracle.normalized_error_grouped(y, ynew, err, rtol, atol, group))
    assert np.array([got]).view(np.int64) == np.array([want]).view(np.int64) or (np.isnan(got) and np.isnan(want))
