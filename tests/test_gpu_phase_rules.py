"""alpha - J and the per-cell norm on each side of the lines between their two kernels, and where
an entry point goes over its cells in several launches, against PyTorch or the same call on fewer
cells, bit for bit."""
import numpy as np
import pytest

from micm_amd import _lib, synthetic
from micm_amd._desc import ARRHENIUS, MechanismDesc

pytestmark = pytest.mark.gpu


def _mech(n_species):
    """Each species decays into the next, the last into nothing."""
    return _lib.Mechanism(MechanismDesc(n_species, [([i], [(i + 1, 0.5)] if i + 1 < n_species else [], ARRHENIUS,
                                                     [1.0, 0.0, 0.0, 300.0, 0.0]) for i in range(n_species)]))


@pytest.mark.parametrize("n_species,cells", [(1, 70), (15, 5000), (16, 5001), (16, 98303), (16, 98304), (16, 163839),
                                             (16, 163840), (29, 163840), (30, 163839), (30, 163841), (30, 327679),
                                             (30, 327680)])
def test_both_kernels(n_species, cells):
    import torch
    print(f"phase rules: {n_species} species, {cells} cells", flush=True)
    mech = _mech(n_species)
    n, nnz = mech.n_species, mech.info.nnz_jacobian
    groups = (cells + 63) // 64
    gen = torch.Generator("cuda").manual_seed(cells)
    rand = lambda v: torch.rand((groups, v, 64), dtype=torch.float64, device="cuda", generator=gen)
    jac, y, ynew, err = rand(nnz), rand(n), rand(n), rand(n) - 0.5
    err[0, 0, :3] = torch.tensor([float("inf"), float("nan"), 0.0])
    atol = torch.rand(n, dtype=torch.float64, device="cuda", generator=gen) * 1e-3 + 1e-6
    last = torch.arange(64, device="cuda") < cells - 64 * (groups - 1)  # the last group's cells

    want = jac.clone()
    want[:, np.asarray(mech.jacobian_diagonal())] += 0.375
    want[-1] = torch.where(last, want[-1], jac[-1])
    mech.alpha_minus_jacobian(cells, jac.data_ptr(), 0.375)
    torch.cuda.synchronize()
    assert torch.equal(jac, want)

    out = torch.full((cells,), -1.0, dtype=torch.float64, device="cuda")
    mech.normalized_error(cells, y.data_ptr(), ynew.data_ptr(), err.data_ptr(), atol.data_ptr(), 1e-4, out.data_ptr())
    q = err / (atol[:, None] + 1e-4 * torch.maximum(y.abs(), ynew.abs()))
    q = q * q
    acc = torch.zeros((groups, 64), dtype=torch.float64, device="cuda")
    for i in range(n):
        acc = acc + q[:, i]
    norm = torch.sqrt(acc / torch.tensor(float(n), dtype=torch.float64, device="cuda"))
    norm = torch.where(norm < 1e-10, torch.full_like(norm, 1e-10), norm).reshape(-1)[:cells]
    assert torch.equal(torch.isnan(out), torch.isnan(norm))
    assert torch.equal(torch.nan_to_num(out, nan=7.0), torch.nan_to_num(norm, nan=7.0))


def test_forcing_in_several_launches():
    """Thirty-two threads a cell: two launches from 2^26 cells on, past one launch's threads from
    2^27."""
    import torch
    mech = _lib.Mechanism(synthetic.readme_mechanism())
    n, r, cells = mech.n_species, mech.n_reactions, (1 << 27) + 70
    if torch.cuda.mem_get_info()[0] < 24 << 30:
        pytest.skip("needs 24 GiB of free device memory")
    print(f"phase rules: forcing of {cells} cells", flush=True)
    groups = (cells + 63) // 64
    gen = torch.Generator("cuda").manual_seed(5)
    y = torch.empty(groups * 64 * n, dtype=torch.float64, device="cuda")
    k = torch.empty(groups * 64 * r, dtype=torch.float64, device="cuda")
    for t in (y, k):
        for part in t.split(1 << 27):
            part.copy_(torch.rand(part.shape, dtype=torch.float64, device="cuda", generator=gen))
    f = torch.full_like(y, -3.0)
    mech.fill_and_add_forcing_terms(cells, k.data_ptr(), y.data_ptr(), f.data_ptr())
    step = 1 << 22
    want = torch.empty(step * n, dtype=torch.float64, device="cuda")
    for c in range(0, cells, step):
        count = min(step, cells - c)
        mech.fill_and_add_forcing_terms(count, k[c * r:].data_ptr(), y[c * n:].data_ptr(), want.data_ptr())
        torch.cuda.synchronize()
        whole, rest = count // 64 * 64, count % 64
        got = f[c * n:]
        assert torch.equal(got[: whole * n], want[: whole * n]), f"cells from {c}"
        if rest:  # the cells of the last group
            a, b = (t[whole * n: (whole + 64) * n].view(n, 64)[:, :rest] for t in (got, want))
            assert torch.equal(a, b)
    del y, k, f, want
    torch.cuda.empty_cache()
