"""The library's choice of kernel by the number of cells, for factors that one wavefront takes in
large numbers: what it names at each side of the line, and that Solves beyond it, in every form
that takes the choice, give the bits of the kernel with the dense block."""
import numpy as np
import pytest

from helpers import bits_equal
from micm_amd import _lib, synthetic

pytestmark = pytest.mark.gpu

LINE = 90112


def _desc(n_species, n_reactions):
    return synthetic.random_mechanism(n_species, n_reactions, {0: n_reactions}, 40 + n_species)


@pytest.mark.parametrize("n_species,n_reactions,changes", [(16, 40, True), (40, 120, True), (50, 150, False),
                                                           (5, 8, False), (12, 40, False)])
def test_default_kernel_by_cells(n_species, n_reactions, changes):
    mech = _lib.Mechanism(_desc(n_species, n_reactions))
    below, at = (mech.cooperative_kernel(4, n_cells=n) for n in (LINE - 1, LINE))
    assert (below != at) == changes
    if changes:
        assert below[0] == _lib.KERNEL_BLOCK and at[0] == _lib.KERNEL_LEVELS and at[1] == 64
    if n_species > 8:  # a requested shape is what was asked for
        assert mech.cooperative_kernel(4, 256, -1, n_cells=LINE) == mech.cooperative_kernel(4, 256, -1)
    with pytest.raises(_lib.MicmHipError):
        mech.cooperative_kernel(4, n_cells=0)


def test_solves_beyond_the_line_are_the_block_kernels():
    desc = _desc(16, 40)
    mech = _lib.Mechanism(desc)
    n = LINE + 37
    print(f"shape rules: {n} cells of 16 species", flush=True)
    cells = synthetic.inputs_60_200(desc, n)
    y0 = np.ascontiguousarray(cells.variables[:, mech.species_order()])
    params = _lib.rosenbrock_parameters(4)

    def solve(form, shape, handoff=-1, recorded=False):
        state = _lib.DeviceState(mech, n)
        state.set_variables(y0)
        state.set_conditions(cells.conditions)
        state.set_cooperative_shape(*shape)
        state.set_handoff(handoff)
        tape = _lib.Tape(mech, n, 2) if recorded else None
        out = []
        for _ in range(2):  # the second in the order of the first's attempts
            if recorded:
                state.solve_recorded(1.0, params, tape, update_rates=True)
            else:
                state.solve(1.0, params, form | _lib.SOLVE_UPDATE_RATES)
            out += [state.get_variables(), *state.results()]
        if recorded:
            out.append(tape.counts())
        return out

    want = solve(_lib.SOLVE_COOPERATIVE, (256, -1))
    for name, got in (("cooperative", solve(_lib.SOLVE_COOPERATIVE, (0, -1))),
                      ("persistent", solve(_lib.SOLVE_PERSISTENT, (0, -1))),
                      ("persistent, hand-off at 2", solve(_lib.SOLVE_PERSISTENT, (0, -1), 2)),
                      ("recorded", solve(None, (0, -1), recorded=True)[:-1])):
        for a, b in zip(got, want):
            assert (bits_equal(a, b) if a.dtype == np.float64 else np.array_equal(a, b)), name
    assert np.array_equal(solve(None, (0, -1), recorded=True)[-1], solve(None, (256, -1), recorded=True)[-1])
