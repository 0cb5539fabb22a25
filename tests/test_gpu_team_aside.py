"""GPU: a march that the device cannot hold steps aside: the stage kernels take over
for the plan, forward, recorded and transposed."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from prince_amd import workloads  # noqa: E402
from prince_amd.solvers.propagation import MultiRHSPropagationSolverETD2  # noqa: E402


def _plan(z, K, team, adjoint=False):
    run = workloads.nuclear_run()
    g = MultiRHSPropagationSolverETD2(z, 0.0, run, K=K)
    g._tuned = {("team", K): team}
    for k, s in enumerate(workloads.batch_sources(run, K, seed=9)):
        g[k].add_source_class(s)
    if adjoint:
        g.set_field_scales(1, np.linspace(0.8, 1.2, K))
    return g, g.prepare(1e-3, with_adjoint=adjoint)


def _oversize(team):
    """More workgroups than any device holds; refused before the launch."""
    team["struct"].nteam, team["struct"].size = 8, 256
    team["struct"].spin_limit = 1


def test_the_stage_kernels_take_over():
    import torch

    g, p = _plan(0.07, 5, False)
    want = g.execute(p).clone()
    g, p = _plan(0.07, 5, True)
    _oversize(p["team"])
    for _ in range(2):
        assert torch.equal(g.execute(p), want)
        assert p["team"] is None and p["graph"] is not None


def test_the_gradient_goes_on_with_the_stage_kernels():
    import torch

    out = []
    for team in (False, True):
        g, p = _plan(0.07, 3, team, adjoint=True)
        if team:
            _oversize(p["team"])
            _oversize(p["team_adjoint"])
        g.forward_checkpointed(p)
        lam = torch.ones_like(p["x"])
        ab = g.adjoint_sweep(p, lam)
        assert p["team"] is None and p.get("team_adjoint") is None
        out.append({k: ab[k].clone() for k in ("lam", "gsrc0", "gsrc1", "gdot")})
    for k, v in out[0].items():
        assert torch.equal(out[1][k], v), k
