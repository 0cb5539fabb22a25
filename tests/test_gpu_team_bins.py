"""GPU: the march bin by bin.  A norm over the whole state hides most of it (84 per
cent of the bins above 1e-30 of a column's peak lie below 1e-10 of the norm), so
columns of every tiling are compared bin by bin with the stage kernels, with the
oracle and with the fixture of the z = 3 batch, over 200 steps and more.

Where a species' spectrum changes sign, a bin can be 1e5 times smaller than the next:
the stencil's rounding is then that of its neighbours (K = 300, two fields, column
195: the stage kernels are 1.2e-7 from the oracle in such a bin, the march 8.8e-8).
Bins below 1e-3 of a neighbour within the stencil's reach are held to the same
tolerance relative to 1e-3 of that neighbour, all others to their own value."""

import numpy as np
import pytest

from oracle.etd2_cpu import OracleETD2
from prince_amd import workloads
from prince_amd.model.photonfields import (
    CMBPhotonSpectrum,
    CombinedPhotonField,
    SyntheticEBL,
)
from prince_amd.solvers.propagation import (
    MultiRHSPropagationSolverETD2,
    UHECRPropagationSolverETD2,
)

from .test_golden import BATCH, load

pytestmark = pytest.mark.gpu

TOL = 1e-8  # bin-wise parity of every other path

# right-hand sides per team: 3-4, 5-8, 9-16, 17-32 and more, odd and even
COLUMNS = [28, 40, 100, 200, 300]


def _scales(K):
    return np.linspace(0.6, 1.4, K)


def _solver(run, z, K, srcs, tuned, scales=None):
    g = MultiRHSPropagationSolverETD2(z, 0.0, run, K=K)
    g._tuned = dict(tuned)
    for k in range(K):
        g[k].add_source_class(srcs[k])
    if scales is not None:
        g.set_field_scales(1, scales)
    return g


def _worst(got, ref, least=100):
    """Largest bin-wise deviation over the columns (arrays [bins][K])."""
    size = np.abs(ref)
    live = size > 1e-30 * size.max(axis=0, keepdims=True)
    assert (live.sum(axis=0) > least).all()
    panels = size.reshape(-1, 64, size.shape[1]) if size.shape[0] % 64 == 0 else size[None]
    scale = panels.copy()
    for o in (1, 2, 3):
        scale[:, o:] = np.maximum(scale[:, o:], 1e-3 * panels[:, :-o])
        scale[:, :-o] = np.maximum(scale[:, :-o], 1e-3 * panels[:, o:])
    return float((np.abs(got - ref)[live] / scale.reshape(size.shape)[live]).max())


@pytest.mark.parametrize("two", [False, True])
@pytest.mark.parametrize("K", COLUMNS)
def test_bins_match_the_stage_kernels(K, two):
    run = workloads.nuclear_run()
    srcs = workloads.batch_sources(run, K, seed=21)
    out = []
    for team in (True, False):
        g = _solver(run, 0.2, K, srcs, {("team", K): team}, _scales(K) if two else None)
        g.solve(1e-3)
        assert (g._plan["team"] is not None) == team
        out.append(g.state.copy())
    worst = _worst(*out)
    print(f"K={K} two={two}: {worst:.2e}")
    assert worst <= TOL


@pytest.mark.parametrize("K", [7, 40, 300])
def test_em_bins_match_the_stage_kernels(K):
    run = workloads.nuclear_em_run()
    srcs = workloads.batch_sources(run, K, seed=22)
    out = []
    for team in (True, False):
        g = _solver(run, 0.2, K, srcs, {("team", K): team})
        g.solve(1e-3)
        assert (g._plan["team"] is not None) == team
        out.append(g.state.copy())
    n, sl = run.dim_states, run.em_slices()[22]
    worst = _worst(out[0][:n], out[1][:n]), _worst(out[0][sl], out[1][sl], 10)
    print(f"K={K}: nuclei {worst[0]:.2e}, photons {worst[1]:.2e}")
    assert max(worst) <= TOL


@pytest.mark.parametrize("K,two", [(3, True), (28, True), (40, False), (100, True), (137, False)])
def test_gradients_match_the_transposed_stages_row_by_row(K, two):
    """Every (species or source slot, column) panel of 64 bins by its own norm."""
    import torch

    run = workloads.nuclear_run()
    srcs = workloads.batch_sources(run, K, seed=23)
    out = []
    for team in (True, False):
        g = _solver(run, 0.2, K, srcs, {("team", K): team}, _scales(K) if two else None)
        p = g.prepare(1e-3, with_adjoint=True)
        assert (p.get("team_adjoint") is not None) == team
        lam = torch.rand(tuple(p["x"].shape), dtype=torch.float64,
                         generator=torch.Generator().manual_seed(4)).to(p["x"].device)
        g.forward_checkpointed(p)
        ab = g.adjoint_sweep(p, lam)
        out.append({k: ab[k].clone() for k in ("lam", "gsrc0", "gsrc1", "gdot")})
        g.close()
    for k in ("lam", "gsrc0", "gsrc1") + (("gdot",) if two else ()):
        diff, ref = (t.norm(dim=-1) for t in (out[0][k] - out[1][k], out[1][k]))
        live = ref > 1e-30 * ref.max()
        assert int(live.sum()) > K
        worst = float((diff[live] / ref[live]).max())
        print(f"K={K} {k}: {worst:.2e}")
        assert worst <= TOL, k


@pytest.mark.parametrize("K", [28, 70, 200, 300])
def test_columns_match_the_oracle(K):
    run = workloads.nuclear_run()
    srcs = workloads.batch_sources(run, K, seed=24)
    g = _solver(run, 0.2, K, srcs, {("team", K): True})
    g.solve(1e-3)
    assert g._plan["team"] is not None
    cols = [0, K // 2 + 1, K - 1]
    o = OracleETD2(0.2, 0.0, run, K=len(cols))
    for i, k in enumerate(cols):
        o.add_source_class(srcs[k], i)
    o.solve(1e-3)
    worst = _worst(g.state[:, cols], o.state)
    print(f"K={K}: {worst:.2e}")
    assert worst <= TOL


@pytest.mark.parametrize("K", [28, 150])
def test_scaled_columns_match_the_oracle(K):
    run = workloads.nuclear_run()
    srcs = workloads.batch_sources(run, K, seed=25)
    scales = _scales(K)
    g = _solver(run, 0.2, K, srcs, {("team", K): True}, scales)
    g.solve(1e-3)
    assert g._plan["team"] is not None
    base = run.photon_field
    amps = base.model_list[1].amplitudes
    try:
        for k in (1, K - 1):
            run.photon_field = CombinedPhotonField(
                [CMBPhotonSpectrum(), SyntheticEBL(amplitudes=amps, scale=scales[k])])
            o = OracleETD2(0.2, 0.0, run)
            o.add_source_class(srcs[k])
            o.solve(1e-3)
            dev = _worst(g.state[:, [k]], o.state.reshape(-1, 1))
            print(f"K={K} scale {scales[k]:.2f}: {dev:.2e}")
            assert dev <= TOL
    finally:
        run.photon_field = base


def test_batch512_march_against_fixture_columns():
    """The z = 3 batch as the default and the autotuner run it now."""
    g = load(BATCH)
    run = workloads.nuclear_run()
    K = int(g["K"])
    srcs = workloads.batch_sources(run, K, seed=int(g["seed"]))
    s = _solver(run, 3.0, K, srcs, {})
    s.solve(dz=1e-3)
    assert s._plan["team"] is not None and s._plan["nwin"] == 288
    dev = _worst(s.state[:, g["columns"]], g["state"], 1000)
    print(f"K=512 march: worst column {dev:.3e}")
    assert dev <= TOL


def test_em_step_graph_equals_direct_launches():
    """The per-step EM kernels, captured and launched one by one (the march stands
    aside for a forced setting only)."""
    run = workloads.proton_em_run()
    states = []
    for graphs in (True, False):
        run.backend.use_hip_graphs = graphs
        try:
            g = UHECRPropagationSolverETD2(0.08, 0.0, run)
            g._tuned = {("team", 1): False}
            g.add_source_class(workloads.proton_source(run))
            g.solve(dz=1e-3)
        finally:
            run.backend.use_hip_graphs = True
        assert g._plan["team"] is None and (g._plan["graph"] is not None) == graphs
        states.append(g.state.copy())
    assert np.array_equal(states[0], states[1])


def test_the_autotuners_choice_matches_a_stage_configuration():
    run = workloads.nuclear_run()
    K = 64
    srcs = workloads.batch_sources(run, K, seed=9)
    g = _solver(run, 0.2, K, srcs, {})
    table = g.autotune(1e-3, steps=5, repeats=1)
    assert any(cfg == {("team", K): True} for _, cfg in table)
    g.solve(1e-3)
    ref = _solver(run, 0.2, K, srcs, {("kt", K): 4})
    ref.solve(1e-3)
    assert ref._plan["team"] is None
    assert _worst(g.state, ref.state) <= TOL
