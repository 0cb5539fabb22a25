"""When the march is taken (no GPU needed): the rule reads the settings of the stage
kernels that it would replace, and of K alone."""

import pytest

from prince_amd.solvers.propagation import ETD2SolverHIP


def _solver(tuned):
    g = object.__new__(ETD2SolverHIP)
    g._tuned = dict(tuned)
    return g


@pytest.mark.parametrize("key", ETD2SolverHIP.STAGE_KEYS)
def test_a_forward_stage_setting_turns_the_forward_march_off(key):
    g = _solver({(key, 64): False})  # any value, the setting is what counts
    assert not g.team_march_for(64) and g.team_march_for(65)
    assert g.adjoint_march_for(64)


@pytest.mark.parametrize("key", ETD2SolverHIP.ADJOINT_STAGE_KEYS)
def test_a_transposed_stage_setting_turns_the_adjoint_march_off(key):
    g = _solver({(key, 64): 4})
    assert not g.adjoint_march_for(64) and g.adjoint_march_for(65)
    assert g.team_march_for(64)


@pytest.mark.parametrize("on", [True, False])
def test_the_explicit_setting_decides_both(on):
    g = _solver({("team", 8): on, ("kt", 8): 4, ("kt_adjoint", 8): 4})
    assert g.team_march_for(8) is on and g.adjoint_march_for(8) is on


def test_settings_of_the_march_itself_and_of_nothing():
    assert _solver({}).team_march_for(7) and _solver({}).adjoint_march_for(7)
    assert _solver({("other", 7): 1}).team_march_for(7)


def test_sizes_at_which_the_stage_kernels_are_faster():
    """Few rows and many columns: a march there is up to nine times slower (7 rows,
    K = 4096).  The explicit setting still decides."""
    g = _solver({})
    for nspec, K in ((1, 512), (1, 4096), (2, 224), (7, 192), (7, 512), (53, 4096), (137, 1024),
                     (305, 1024)):
        assert not g.team_march_for(K, nspec), (nspec, K)
        assert _solver({("team", K): True}).team_march_for(K, nspec)
    for nspec, K in ((1, 1), (1, 448), (2, 256), (7, 128), (53, 64), (89, 300), (305, 1), (305, 512)):
        assert g.team_march_for(K, nspec), (nspec, K)
    for nspec, K, on in ((305, 128, True), (305, 512, False), (7, 64, True), (7, 128, False)):
        assert g.team_march_for(K, nspec, 2) is on
    assert g.team_march_for(1024, 305, 1, gradient=True)
    for nspec, K, on in ((305, 128, True), (305, 256, False), (17, 256, True), (2, 128, False)):
        assert g.adjoint_march_for(K, nspec, 2) is on
    for nspec, K, on in ((305, 1024, True), (2, 512, True), (2, 768, False)):
        assert g.adjoint_march_for(K, nspec, 1) is on
