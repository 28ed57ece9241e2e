"""Single phases on more cells than one launch has threads for when a cell takes as many as the
kernels for few cells give it (the per-cell norm sixteen, alpha - J one per species; a launch of
2^32 threads and more runs their number modulo 2^32).  Outputs against the same operations in
PyTorch, bit for bit, over every cell."""
import numpy as np
import pytest

from micm_amd import _lib, synthetic
from micm_amd._desc import ARRHENIUS, MechanismDesc

pytestmark = pytest.mark.gpu

GIB = 1 << 30


def _free(gib):
    import torch
    if torch.cuda.mem_get_info()[0] < gib * GIB:
        pytest.skip(f"needs {gib} GiB of free device memory")


def test_normalized_error_of_many_cells():
    import torch
    _free(24)
    mech = _lib.Mechanism(synthetic.readme_mechanism())
    n, cells = mech.n_species, (1 << 28) + 37
    groups = (cells + 63) // 64
    print(f"normalized error: {cells} cells of {n} species", flush=True)
    gen = torch.Generator("cuda").manual_seed(7)
    y = torch.zeros(groups * n * 64, dtype=torch.float64, device="cuda")  # also the new values
    err = torch.empty_like(y)
    for part in err.split(1 << 27):
        part.copy_(torch.rand(part.shape, dtype=torch.float64, device="cuda", generator=gen))
    atol = torch.full((n,), 1e-3, dtype=torch.float64, device="cuda")
    out = torch.full((cells,), -1.0, dtype=torch.float64, device="cuda")
    mech.normalized_error(cells, y.data_ptr(), y.data_ptr(), err.data_ptr(), atol.data_ptr(), 1e-6, out.data_ptr())
    torch.cuda.synchronize()
    step = 1 << 20  # groups
    # (divisors on the device: PyTorch multiplies by the inverse of a number)
    count = torch.tensor(float(n), dtype=torch.float64, device="cuda")
    for g in range(0, groups, step):
        q = err.view(groups, n, 64)[g: g + step] / atol[0]
        q = q * q
        want = q[:, 0]
        for i in range(1, n):
            want = want + q[:, i]
        want = torch.clamp(torch.sqrt(want / count), min=1e-10).reshape(-1)
        got = out[g * 64: (g + step) * 64]
        wrong = int((got != want[: got.numel()]).sum())
        assert wrong == 0, f"{wrong} cells of the groups from {g}"
    del y, err, out
    torch.cuda.empty_cache()


def test_alpha_minus_jacobian_of_many_cells():
    import torch
    _free(48)
    desc = MechanismDesc(8, [([0], [(1, 1.0)], ARRHENIUS, [1.0, 0.0, 0.0, 300.0, 0.0])])
    mech = _lib.Mechanism(desc)
    n, nnz, cells = mech.n_species, mech.info.nnz_jacobian, (1 << 29) + 37
    groups = (cells + 63) // 64
    print(f"alpha - J: {cells} cells of {n} species, {nnz} elements", flush=True)
    jac = torch.zeros(groups * nnz * 64, dtype=torch.float64, device="cuda")
    mech.alpha_minus_jacobian(cells, jac.data_ptr(), 0.75)
    torch.cuda.synchronize()
    want = torch.zeros(nnz, 1, dtype=torch.float64, device="cuda")
    want[np.asarray(mech.jacobian_diagonal())] = 0.75
    view, step = jac.view(groups, nnz, 64), 1 << 20
    for g in range(0, groups - 1, step):
        part = view[g: min(g + step, groups - 1)]
        wrong = int((part != want).sum())
        assert wrong == 0, f"{wrong} elements of the groups from {g}"
    last = view[groups - 1]
    assert torch.equal(last[:, :37], want.expand(nnz, 37)) and not last[:, 37:].any()
    del jac, view, last, part
    torch.cuda.empty_cache()
