"""The cooperative kernel with the factor's dense block (k_coop_tail) against the reference's
arithmetic, bit for bit, at the sizes where its layout changes: a block of the whole
mechanism (16 species), one row outside it, one row past a sixteen, a full wavefront of rows
and one more, and the largest mechanism it takes (a species for each of its 256 threads).  Some
cells start from values whose rates overflow, so that their factors hold infinities and the
block is done again with its products tested."""
import numpy as np
import pytest

from helpers import bits_equal, dev, dev_zeros, host
from micm_amd import _lib, synthetic
from oracle import OraclePortableMath

pytestmark = pytest.mark.gpu

SIZES = [(16, 30), (17, 40), (33, 90), (48, 140), (64, 170), (65, 180), (129, 340), (256, 700)]


@pytest.mark.parametrize("stage", [5, 6])
@pytest.mark.parametrize("n_species,n_reactions", SIZES)
def test_block_kernel_matches_reference_math(n_species, n_reactions, stage):
    print(f"tail: {n_species} species, {n_reactions} reactions, stage {stage}", flush=True)
    desc = synthetic.random_mechanism(n_species, n_reactions, {0: n_reactions}, 100 + n_species)
    n = 24
    cells = synthetic.inputs_60_200(desc, n)
    cells.variables[-8:] *= np.array([1e60, 1e90, 1e120, 1e150, 1e200, 1e250, 1e290, 1e300])[:, None]
    mech = _lib.Mechanism(desc)
    y0 = cells.variables[:, mech.species_order()]
    state = _lib.DeviceState(mech, n)
    state.set_variables(y0)
    state.set_conditions(cells.conditions)
    state.update_state_parameters()
    state.set_cooperative_shape(256, stage)
    tableau, dt = (4, 300.0) if stage == 6 else (3, 60.0)
    state.solve(dt, _lib.rosenbrock_parameters(tableau), _lib.SOLVE_COOPERATIVE)
    oracle = OraclePortableMath(desc, tableau)
    y, status, stats, _ = oracle.solve(cells.conditions, cells.custom, y0, dt, 1)
    got_status, got_stats, _ = state.results()
    assert np.array_equal(got_status, status) and np.array_equal(got_stats, stats)
    assert bits_equal(state.get_variables(), y)
    assert (status[-8:] != 2).any()  # some of the large cells do leave the finite range


@pytest.mark.parametrize("kind", ["negative_zero", "infinite", "lower_diagonal"])
@pytest.mark.parametrize("n_species,n_reactions", [(16, 30), (33, 90), (65, 180), (129, 340)])
def test_block_phases_take_every_operand(n_species, n_reactions, kind):
    """The single-phase LU and substitution with the block on what its unmasked products must not
    see: -0 in the matrix and the right-hand side, infinities, and a lower diagonal that is not 1."""
    print(f"tail phases: {n_species} species, {kind}", flush=True)
    desc = synthetic.random_mechanism(n_species, n_reactions, {0: n_reactions}, 300 + n_species)
    n = 70
    cells = synthetic.inputs_60_200(desc, n)
    mech, oracle = _lib.Mechanism(desc), OraclePortableMath(desc, 4)
    N = mech.n_species
    y0 = cells.variables[:, mech.species_order()]
    k = oracle.rate_constants(cells.conditions, cells.custom)
    jac, x = oracle.jacobian(k, y0), oracle.forcing(k, y0)
    rng = np.random.default_rng(n_species)
    if kind == "negative_zero":
        jac[rng.random(jac.shape) < 0.2] = -0.0
        x[rng.random(x.shape) < 0.3] = -0.0
    diag = mech.jacobian_diagonal()
    jac[:, diag] += 0.25  # every pivot away from zero
    if kind == "infinite":
        jac[np.arange(n), rng.integers(0, jac.shape[1], n)] = np.inf
        x[::3, rng.integers(0, N)] = -np.inf
    _, lower, upper = oracle.lu(jac, 0.0)
    dj, dl, du, dx = dev(jac), dev_zeros(n, mech.nnz_lower), dev_zeros(n, mech.nnz_upper), dev(x)
    mech.lu_decompose(n, dj.data_ptr(), dl.data_ptr(), du.data_ptr())
    same = lambda a, b: np.all((a.view(np.int64) == b.view(np.int64)) | (np.isnan(a) & np.isnan(b)))
    assert same(host(dl, n, mech.nnz_lower), lower) and same(host(du, n, mech.nnz_upper), upper)
    if kind == "lower_diagonal":
        rows, cols = mech.patterns()["lower"]
        lower[:, rows == cols] = rng.uniform(0.5, 2.0, (n, N))
        dl = dev(lower)
    want = oracle.lu_solve(lower, upper, x)
    mech.lu_solve(n, dl.data_ptr(), du.data_ptr(), dx.data_ptr())
    assert same(host(dx, n, N), want)
