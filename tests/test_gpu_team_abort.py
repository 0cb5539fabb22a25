"""GPU: a march whose wait between workgroups gives up.  The tiny limit on the waits
makes that happen at once (every kernel still ends by itself); whatever the
workgroups had stored by then, no result the caller sees may be finite."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from prince_amd import workloads  # noqa: E402
from prince_amd.solvers.propagation import MultiRHSPropagationSolverETD2  # noqa: E402


def _solver(run, z, K, scales=None):
    g = MultiRHSPropagationSolverETD2(z, 0.0, run, K=K)
    g._tuned = {("team", K): True}
    for k, s in enumerate(workloads.batch_sources(run, K, seed=2)):
        g[k].add_source_class(s)
    if scales is not None:
        g.set_field_scales(1, scales)
    return g


def _none_finite(t):
    return not bool(t.isfinite().any())


@pytest.mark.parametrize("K", [1, 9, 40])
def test_an_aborted_march_leaves_nothing_finite(K):
    import torch

    g = _solver(workloads.nuclear_run(), 0.02, K)
    p = g.prepare(1e-3)
    want = g.execute(p).clone()
    p["team"]["struct"].spin_limit = 1
    assert _none_finite(g.execute(p))
    p["team"]["struct"].spin_limit = 0
    assert torch.equal(g.execute(p), want)


def test_photons_of_an_aborted_range_are_not_finite():
    """In the last range of two: the photons follow from its Bethe-Heitler sums."""
    g = _solver(workloads.nuclear_em_run(), 0.3, 3)
    p = g.prepare(1e-3)
    x = g.execute(p, 0, g.EM_RANGE)
    assert bool(x.isfinite().all())
    p["team"]["struct"].spin_limit = 1
    assert _none_finite(g.execute(p, g.EM_RANGE, p["nsteps"]))
    gam = g.em_host_state(p)[2 * g.prince_run.em_grid.d:]
    assert not np.isfinite(gam).any()


@pytest.mark.parametrize("which", ["recompute", "first chunk", "last chunk"])
def test_an_aborted_gradient_is_not_finite(which):
    import torch

    K = 5
    g = _solver(workloads.nuclear_run(), 0.1, K, np.linspace(0.7, 1.3, K))
    p = g.prepare(1e-3, with_adjoint=True)
    lam = torch.ones_like(p["x"])
    g.forward_checkpointed(p)
    g.adjoint_sweep(p, lam)  # finite accumulators from before
    last = p["nsteps"] - p["nsteps"] % p["ckpt_chunk"]
    run, adjoint = g._team_run, g._team_adjoint_run

    def team_run(plan, st, k0, k1):
        plan["team"]["struct"].spin_limit = int(which == "recompute" and k0 == 0)
        return run(plan, st, k0, k1)

    def team_adjoint_run(plan, k0, k1):
        at = {"first chunk": last, "last chunk": 0}.get(which, -1)
        plan["team_adjoint"]["struct"].spin_limit = int(k0 == at)
        return adjoint(plan, k0, k1)

    g._team_run, g._team_adjoint_run = team_run, team_adjoint_run
    ab = g.adjoint_sweep(p, lam)
    # the sweep itself does not read the recorded states, the EBL-scale gradient does
    names = ("gdot",) if which == "recompute" else ("lam", "gdot", "gsrc0", "gsrc1")
    for k in names:
        assert _none_finite(ab[k]), k
