"""The kernel with one cell per lane on each side of the line from which mechanisms with more
reactions or species take it, against a workgroup per cell (a requested staging), bit for bit: both
builds of the kernel, values that leave the finite range, a second Solve, and every form that
routes to it."""
import numpy as np
import pytest

from helpers import bits_equal
from micm_amd import _lib
from micm_amd._desc import ARRHENIUS, MechanismDesc

pytestmark = pytest.mark.gpu

LINE = 2304


def _mechanism(n_species, n_reactions):
    rng = np.random.default_rng(31 * n_species + n_reactions)
    reactions = []
    for r in range(n_reactions):
        reactants = [int(s) for s in rng.integers(0, n_species, 1 + r % 2)]
        products = [(int(rng.integers(0, n_species)), float(rng.uniform(0.1, 0.5)))]
        reactions.append((reactants, products, ARRHENIUS, [float(10.0 ** rng.uniform(-4, -1)), 0.0, 0.0, 300.0, 0.0]))
    return MechanismDesc(n_species, reactions, ignore_unused_species=True)


@pytest.mark.parametrize("n_species,n_reactions,tableau", [(2, 24, 4), (4, 18, 3), (5, 8, 4), (5, 12, 3), (6, 4, 3),
                                                           (7, 3, 2)])
@pytest.mark.parametrize("n_cells", [LINE - 1, LINE, LINE + 65])
def test_lane_kernel_beyond_its_line(n_species, n_reactions, tableau, n_cells):
    print(f"tiny rules: {n_species} species, {n_reactions} reactions, {n_cells} cells", flush=True)
    mech = _lib.Mechanism(_mechanism(n_species, n_reactions))
    params = _lib.rosenbrock_parameters(tableau)
    kernel = mech.cooperative_kernel(params.stages, n_cells=n_cells)[0]
    assert (kernel == _lib.KERNEL_LANE) == (n_cells >= LINE)
    y0 = np.random.default_rng(n_cells).uniform(0.1, 2.0, (n_cells, mech.n_species))
    y0[-40:] *= np.logspace(40, 300, 40)[:, None]

    def solve(form, shape, handoff=-1):
        state = _lib.DeviceState(mech, n_cells)
        state.set_variables(y0)
        state.set_conditions(np.tile([280.0, 9e4, 38.0], (n_cells, 1)))
        state.set_cooperative_shape(*shape)
        state.set_handoff(handoff)
        out = []
        for _ in range(2):
            state.solve(40.0, params, form | _lib.SOLVE_UPDATE_RATES)
            out += [state.get_variables(), *state.results()]
        return out

    want = solve(_lib.SOLVE_COOPERATIVE, (64, 0))
    for name, got in (("cooperative", solve(_lib.SOLVE_COOPERATIVE, (0, -1))),
                      ("cooperative, 128 threads", solve(_lib.SOLVE_COOPERATIVE, (128, -1))),
                      ("persistent", solve(_lib.SOLVE_PERSISTENT, (0, -1))),
                      ("persistent, hand-off at 2", solve(_lib.SOLVE_PERSISTENT, (0, -1), 2))):
        for a, b in zip(got, want):
            same = np.array_equal(a, b) if a.dtype != np.float64 else \
                (bits_equal(a, b) or np.all((a.view(np.int64) == b.view(np.int64)) | (np.isnan(a) & np.isnan(b))))
            assert same, name
