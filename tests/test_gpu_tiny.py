"""Solves of mechanisms of at most eight species, one cell per lane (k_tiny), against the
reference's arithmetic, bit for bit: every number of species it takes and the first it does not,
cells around a wavefront, each form that routes to it, cells handed to it part way, and cells
whose values leave the finite range."""
import numpy as np
import pytest

from helpers import bits_equal
from micm_amd import _lib, synthetic
from micm_amd._desc import ARRHENIUS, MechanismDesc
from oracle import OraclePortableMath

pytestmark = pytest.mark.gpu


def _mechanism(n_species):
    """Reactions of one to three reactants (repeats among them), products of any species."""
    rng = np.random.default_rng(n_species)
    reactions = []
    for r in range(2 * n_species):
        reactants = [int(s) for s in rng.integers(0, n_species, 1 + r % 3)]
        products = [(int(rng.integers(0, n_species)), float(rng.uniform(0.1, 0.9))) for _ in range(int(rng.integers(0, 4)))]
        reactions.append((reactants, products, ARRHENIUS, [float(10.0 ** rng.uniform(-4, 0)), 0.0, 0.0, 300.0, 0.0]))
    return MechanismDesc(n_species, reactions, ignore_unused_species=True)


def _cells(n_species, n, large):
    rng = np.random.default_rng(100 + n_species)
    y = rng.uniform(0.0, 2.0, (n, n_species))
    if large:
        y[n // 2:] *= np.logspace(40, 300, n - n // 2)[:, None]
    return synthetic.CellInputs(np.tile([280.0, 9e4, 38.0], (n, 1)), y, np.zeros((n, 0)))


def _check(mech, desc, cells, form, tableau, dt, handoff=-1, shape=(0, -1), group=1, update=False):
    y0 = cells.variables[:, mech.species_order()]
    state = _lib.DeviceState(mech, cells.n_cells)
    state.set_variables(y0)
    state.set_conditions(cells.conditions)
    state.set_cooperative_shape(*shape)
    state.set_handoff(handoff)
    state.set_lockstep_order(group)
    params = _lib.rosenbrock_parameters(tableau)
    total = 0
    for _ in range(2):
        state.update_state_parameters()
        state.solve(dt, params, form)
        total = total + state.results()[1]
    lockstep = group if form == _lib.SOLVE_LOCKSTEP else False
    y, status, stats, ft = OraclePortableMath(desc, tableau).solve(cells.conditions, cells.custom, y0, dt, 2,
                                                                   lockstep=lockstep)
    got_status, _, got_ft = state.results()
    assert np.array_equal(got_status, status) and np.array_equal(total, stats)
    assert bits_equal(got_ft, ft) and bits_equal(state.get_variables(), y)


@pytest.mark.parametrize("n_species", [1, 2, 3, 4, 5, 7, 8, 9])
@pytest.mark.parametrize("n_cells,large", [(1, False), (65, False), (130, True)])
def test_per_cell_steps(n_species, n_cells, large):
    print(f"tiny: {n_species} species, {n_cells} cells", flush=True)
    desc = _mechanism(n_species)
    mech = _lib.Mechanism(desc)
    cells = _cells(mech.n_species, n_cells, large)
    _check(mech, desc, cells, _lib.SOLVE_COOPERATIVE, 4, 30.0)
    _check(mech, desc, cells, _lib.SOLVE_COOPERATIVE, 3, 30.0, shape=(128, -1))
    _check(mech, desc, cells, _lib.SOLVE_PERSISTENT, 61, 30.0)
    _check(mech, desc, cells, _lib.SOLVE_PERSISTENT, 2, 30.0, handoff=2)


@pytest.mark.parametrize("n_species", [1, 3, 4, 5, 8, 9])
@pytest.mark.parametrize("n_cells,group", [(1, 1), (2, 4), (63, 1), (64, 4), (64, 64), (65, 1)])
def test_one_step_size(n_species, n_cells, group):
    print(f"tiny lockstep: {n_species} species, {n_cells} cells, order {group}", flush=True)
    desc = _mechanism(n_species)
    mech = _lib.Mechanism(desc)
    _check(mech, desc, _cells(mech.n_species, n_cells, False), _lib.SOLVE_LOCKSTEP, 3, 30.0, group=group)
    _check(mech, desc, _cells(mech.n_species, n_cells, n_cells > 1), _lib.SOLVE_LOCKSTEP, 4, 30.0, group=group)
