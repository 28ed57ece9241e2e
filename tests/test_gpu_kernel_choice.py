"""micm_hip_mechanism_cooperative_kernel at the edges of the kernels' ranges of species."""
import pytest

from micm_amd import _lib, synthetic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_species,default", [(2, _lib.KERNEL_LANE), (5, _lib.KERNEL_LANE), (8, _lib.KERNEL_LEVELS), (9, _lib.KERNEL_LEVELS),
                                               (15, _lib.KERNEL_LEVELS), (16, _lib.KERNEL_BLOCK),
                                               (256, _lib.KERNEL_BLOCK), (257, _lib.KERNEL_LEVELS)])
def test_kernel_of_a_shape(n_species, default):
    reactions = 3 * n_species // 2
    desc = synthetic.random_mechanism(n_species, reactions, {0: reactions}, 70 + n_species)
    mech = _lib.Mechanism(desc)
    print(f"kernel choice: {n_species} species", flush=True)
    if default == _lib.KERNEL_LEVELS and not mech.cooperative_supported(4):
        default = _lib.KERNEL_NONE
    # (the lane takes 5 species from 2,304 cells on)
    if n_species == 5:
        assert mech.cooperative_kernel(4, n_cells=2303)[0] == _lib.KERNEL_LEVELS
    kernel, threads, _, waves = mech.cooperative_kernel(4, n_cells=2304)
    assert kernel == default
    assert (waves in (2, 3)) == (kernel == _lib.KERNEL_BLOCK)
    assert threads == {_lib.KERNEL_LANE: 0, _lib.KERNEL_NONE: 0, _lib.KERNEL_BLOCK: 256, _lib.KERNEL_LEVELS: 64}[kernel]
    three, two, seven = (mech.cooperative_kernel(4, 256, stage) for stage in (5, 6, 7))
    assert two == seven
    if default == _lib.KERNEL_BLOCK:
        assert three[3] == 3 and two[3] == 2
        assert mech.cooperative_kernel(4, 256, -1) == mech.cooperative_kernel(4, 256, 4) == mech.cooperative_kernel(4)
    else:
        assert three == two and two[0] not in (_lib.KERNEL_BLOCK, _lib.KERNEL_LANE)
    for stages, threads, stage in ((0, 0, -1), (7, 0, -1), (4, 65, -1), (4, 0, 8), (4, 0, -2)):
        with pytest.raises(_lib.MicmHipError):
            mech.cooperative_kernel(stages, threads, stage)
