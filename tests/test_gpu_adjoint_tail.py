"""The adjoint's reverse sweep with the factor's dense block (k_adjoint_tail) against the oracle's
adjoint at the sizes where its layout changes, with reactions of one to four reactants (the
second derivatives its lists pack) and one of five (which its lists cannot hold)."""
import numpy as np
import pytest

from micm_amd import _lib, synthetic
from micm_amd._desc import ARRHENIUS, MechanismDesc
from oracle import OraclePortableMath
from test_gpu_adjoint import _adjoint, _host_tape, _record, _smooth_cells

pytestmark = pytest.mark.gpu

SIZES = [(16, 30), (17, 40), (33, 90), (48, 140), (64, 170), (65, 180), (129, 340)]


def _mechanism(n_species, n_reactions, most, seed):
    """Reactions of 1 .. most reactants (repeats among them) of order-one rates; products above
    their highest reactant, so that nothing grows."""
    rng = np.random.default_rng(seed)
    reactions = []
    for r in range(n_reactions):
        n_react = 1 + r % most
        reactants = [int(s) for s in rng.integers(0, n_species - 1, n_react)]
        lowest = max(reactants) + 1
        products = [(int(rng.integers(lowest, n_species)), float(rng.uniform(0.1, 1.0)))
                    for _ in range(int(rng.integers(1, 4)))]
        reactions.append((reactants, products, ARRHENIUS, [float(rng.uniform(1e-4, 1e-2)), 0.0, 0.0, 300.0, 0.0]))
    return MechanismDesc(n_species, reactions)


@pytest.mark.parametrize("tableau", [2, 4])
@pytest.mark.parametrize("n_species,n_reactions,most", [(*s, 4) for s in SIZES] + [(256, 400, 2), (20, 60, 5)])
def test_reverse_sweep_matches_oracle(n_species, n_reactions, most, tableau):
    print(f"adjoint: {n_species} species, up to {most} reactants, {tableau} stages", flush=True)
    desc = _mechanism(n_species, n_reactions, most, n_species)
    n, dt = 20, 100.0
    rng = np.random.default_rng(n_species + 1)
    cells = synthetic.CellInputs(np.tile([280.0, 9e4, 38.0], (n, 1)), rng.uniform(0.1, 1.0, (n, n_species)),
                                 np.zeros((n, 0)))
    mech = _lib.Mechanism(desc)
    state, tape, params = _record(mech, cells, tableau, dt, 2, 2004, atol=1e-10)
    assert tape.overflowed() == 0 and _smooth_cells(tape, dt).all()
    lam = rng.standard_normal((n, n_species))
    gy, gk = _adjoint(state, tape, params, lam)
    o = OraclePortableMath(desc, tableau)
    gy_ref, gk_ref = o.adjoint(state.get_rate_constants(), _host_tape(tape), lam)
    # both sum in 64 bits in orders of their own: normwise, as the adjoint of the recorded
    # map is compared everywhere
    for a, b in ((gy, gy_ref), (gk, gk_ref)):
        scale = np.abs(b).max(axis=1)
        assert (scale > 0).all() and np.all(np.abs(a - b).max(axis=1) <= 1e-9 * scale)


@pytest.mark.parametrize("n_species,n_reactions", [(16, 30), (33, 90), (65, 180)])
def test_values_that_are_not_finite_stay_in_their_columns(n_species, n_reactions):
    """A NaN in one cell's seed reaches the entries that the fill pattern takes it to and no others:
    the block's structural zeros are not multiplied with it."""
    print(f"adjoint, NaN seed: {n_species} species", flush=True)
    desc = _mechanism(n_species, n_reactions, 2, n_species)
    n = 20
    rng = np.random.default_rng(n_species + 2)
    cells = synthetic.CellInputs(np.tile([280.0, 9e4, 38.0], (n, 1)), rng.uniform(0.1, 1.0, (n, n_species)),
                                 np.zeros((n, 0)))
    mech = _lib.Mechanism(desc)
    state, tape, params = _record(mech, cells, 4, 100.0, 1, 1002, atol=1e-10)
    lam = rng.standard_normal((n, n_species))
    for c in range(n):
        if c % 4:
            lam[c, rng.integers(n_species)] = np.nan
    gy, gk = _adjoint(state, tape, params, lam)
    o = OraclePortableMath(desc, 4)
    gy_ref, gk_ref = o.adjoint(state.get_rate_constants(), _host_tape(tape), lam)
    for a, b in ((gy, gy_ref), (gk, gk_ref)):
        keep = np.isfinite(b)
        assert np.array_equal(np.isfinite(a), keep)
        scale = np.abs(np.where(keep, b, 0.0)).max(axis=1, keepdims=True)
        assert np.all((np.abs(a - b) <= 1e-9 * scale) | ~keep)
