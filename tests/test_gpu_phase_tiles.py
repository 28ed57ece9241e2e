"""The single-phase LU and substitution against the reference's arithmetic, bit for bit, on sparse
factors around the lines between the kernel with the dense block and the tiled ones (tiles of four
and two cells among them), and on mechanisms of more than 129 species, up to and past the 256 that
the Solve's kernel with the block takes."""
import numpy as np
import pytest

from helpers import bits_equal, dev, dev_zeros, host
from micm_amd import _lib, synthetic
from oracle import OraclePortableMath

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_species,n_reactions,n_cells", [
    (160, 170, 70), (160, 170, 769), (200, 200, 771), (200, 200, 2049), (256, 256, 775), (257, 260, 70),
    (300, 310, 770), (400, 400, 129)])
def test_phases_of_sparse_factors(n_species, n_reactions, n_cells):
    desc = synthetic.random_mechanism(n_species, n_reactions, {0: n_reactions}, 5)
    mech, oracle = _lib.Mechanism(desc), OraclePortableMath(desc, 4)
    i, N = mech.info, mech.n_species
    print(f"phase tiles: {n_species} species, {i.nnz_lower + i.nnz_upper - N} entries, {i.lu_multiply_adds} products, "
          f"{n_cells} cells", flush=True)
    cells = synthetic.inputs_60_200(desc, n_cells)
    y = cells.variables[:, mech.species_order()]
    k = oracle.rate_constants(cells.conditions, cells.custom)
    jac, x = oracle.jacobian(k, y), oracle.forcing(k, y)
    a, lower, upper = oracle.lu(jac, 0.25)
    want = oracle.lu_solve(lower, upper, x)
    dj, dl, du, dx = dev(a), dev_zeros(n_cells, mech.nnz_lower), dev_zeros(n_cells, mech.nnz_upper), dev(x)
    mech.lu_decompose(n_cells, dj.data_ptr(), dl.data_ptr(), du.data_ptr())
    assert bits_equal(host(dl, n_cells, mech.nnz_lower), lower) and bits_equal(host(du, n_cells, mech.nnz_upper), upper)
    mech.lu_solve(n_cells, dl.data_ptr(), du.data_ptr(), dx.data_ptr())
    assert bits_equal(host(dx, n_cells, N), want)
