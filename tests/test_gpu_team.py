"""GPU: the team march (one cooperative launch per step range) against the
per-stage kernels: every column tiling of its dispatch, recorded steps, two photon
fields, partial ranges, and the conditions under which it steps aside."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from prince_amd import workloads  # noqa: E402
from prince_amd.solvers.propagation import (  # noqa: E402
    MultiRHSPropagationSolverETD2,
    UHECRPropagationSolverETD2,
)


def _solver(run, z, K, seed, team, scales=None):
    g = MultiRHSPropagationSolverETD2(z, 0.0, run, K=K)
    g._tuned = {("team", K): team}
    for k, s in enumerate(workloads.batch_sources(run, K, seed=seed)):
        g[k].add_source_class(s)
    if scales is not None:
        g.set_field_scales(1, scales)
    return g


def _norm_dev(a, b):
    return float((a - b).norm() / b.norm())


# sums of up to 2500 positive products per entry in another order, over 2 z / dz
# stages: 2500 eps per stage at most, 5e-13 x 200 stages = 1e-10 (norm-wise)
TOL = 1e-10


@pytest.mark.parametrize("two", [False, True])
@pytest.mark.parametrize("K", [1, 2, 8, 9, 16, 17, 33, 70, 137, 300])
def test_march_equals_stage_kernels(K, two):
    """K around every edge of the tiling: 1, 2, 3-4, 5-8, 9-16, 17-32 and more
    right-hand sides per team, odd counts, empty teams."""
    run = workloads.nuclear_run()
    scales = np.linspace(0.6, 1.4, K) if two else None
    out = []
    for team in (True, False):
        g = _solver(run, 0.05, K, 3, team, scales)
        p = g.prepare(1e-3)
        assert (p["team"] is not None) == team
        x = g.execute(p).clone()
        assert bool(np.isfinite(float(x.sum())))
        assert bool((g.execute(p) == x).all())  # the same bits again
        out.append(x)
        g.close()
    dev = _norm_dev(*out)
    print(f"K={K} two={two}: {dev:.2e}")
    assert dev <= TOL


def test_march_in_pieces_and_records():
    """Steps [0, 37) then [37, n): the same bits as one march; recorded stage
    vectors equal the state's own history."""
    import ctypes

    import torch

    from prince_amd import _lib

    run = workloads.nuclear_run()
    g = _solver(run, 0.06, 5, 4, True)
    p = g.prepare(1e-3)
    whole = g.execute(p).clone()
    g.execute(p, 0, 37)
    x37 = p["x"].clone()
    g.execute(p, 37, p["nsteps"])
    assert torch.equal(p["x"], whole)
    rec = torch.zeros((4, 3) + tuple(whole.shape), dtype=torch.float64, device=whole.device)
    st = _lib.PrhState(x=p["x"].data_ptr(), a=p["bufs"]["a"].data_ptr(),
                       fphi=p["bufs"]["fphi"].data_ptr(), rec_x=rec[0].data_ptr(),
                       rec_a=rec[1].data_ptr(), rec_fx=rec[2].data_ptr(),
                       rec_fa=rec[3].data_ptr(), rec_first=37, rec_count=3)
    p["x"].copy_(x37)
    assert g._team_run(p, st, 37, 40)
    assert torch.equal(rec[0, 0], x37)
    ref = torch.zeros_like(rec)
    st2 = _lib.PrhState(x=p["x"].data_ptr(), a=p["bufs"]["a"].data_ptr(),
                        fphi=p["bufs"]["fphi"].data_ptr(), rec_x=ref[0].data_ptr(),
                        rec_a=ref[1].data_ptr(), rec_fx=ref[2].data_ptr(),
                        rec_fa=ref[3].data_ptr(), rec_first=37, rec_count=3,
                        dpart=p["bufs"]["dpart"].data_ptr())
    p["x"].copy_(x37)
    _lib.check(g._lib.prh_etd2_steps(ctypes.byref(p["op"]), ctypes.byref(p["sch"]),
                                     ctypes.byref(st2), 37, 40, p["stream"]), "steps")
    for i in range(4):
        assert _norm_dev(rec[i], ref[i]) <= TOL, i


def test_a_nan_column_stays_in_its_column():
    """Columns share waves; a column of NaN (or infinities) must not reach its
    neighbours, whatever half of a wave they sit in."""
    import torch

    run = workloads.nuclear_run()
    for K in (2, 7, 40):
        g = _solver(run, 0.02, K, 6, True)
        p = g.prepare(1e-3)
        good = g.execute(p).clone()
        for bad in (float("nan"), float("inf")):
            p["x"].zero_()
            p["x"][:, 1, :] = bad
            g.fold_windows(p)
            g._launch_steps(p, 0, p["nsteps"])
            keep = [k for k in range(K) if k != 1]
            assert torch.equal(p["x"][:, keep], good[:, keep]), (K, bad)
            assert not bool(torch.isfinite(p["x"][:, 1]).any())
        g.close()


def test_forced_stage_configuration_runs_the_stage_kernels():
    run = workloads.proton_run()
    g = UHECRPropagationSolverETD2(0.1, 0.0, run)
    g.add_source_class(workloads.proton_source(run))
    g.solve(1e-3)
    assert g._plan["team"] is not None and g._plan["graph"] is None
    ref = g.state.copy()
    g._tuned = {("kt", 1): 1}
    g.solve(1e-3)
    assert g._plan["team"] is None
    # one row, one term order: rounding of the fused products only
    assert np.linalg.norm(g.state - ref) <= 1e-12 * np.linalg.norm(ref)


def test_a_capturing_stream_takes_the_stage_kernels():
    """Inside a stream capture the march steps aside; replays equal the direct run."""
    import torch

    run = workloads.nuclear_run()
    g = _solver(run, 0.01, 3, 8, True)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        p = g.prepare(1e-3)
        want = g.execute(p).clone()
        graph = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=side):
            p["x"].zero_()
            g._launch_steps(p, 0, p["nsteps"])
        assert p["team"] is not None
        for _ in range(3):
            p["x"].fill_(1.0)
            graph.replay()
            torch.cuda.synchronize()
            assert _norm_dev(p["x"], want) <= TOL


@pytest.mark.parametrize("K,z", [(1, 0.03), (3, 0.021), (16, 0.02), (17, 0.02), (70, 0.3)])
def test_em_march_equals_the_stage_kernels(K, z):
    """Nuclei and photons of the march with the EM cascade against the per-step EM
    kernels: odd step counts (the photon buffers alternate), ragged columns of the
    16-column photon tiles, and more steps than one range."""
    run = workloads.nuclear_em_run()
    out = []
    for team in (True, False):
        g = _solver(run, z, K, 5, team)
        p = g.prepare(1e-3)
        assert (p["team"] is not None) == team
        x = g.execute(p).clone()
        gam = g.em_host_state(p).copy()
        assert bool((g.execute(p) == x).all()) and np.array_equal(g.em_host_state(p), gam)
        if team and z > 0.25:
            assert p["nsteps"] > g.EM_RANGE
            g.execute(p, 0, 111)
            g.execute(p, 111, p["nsteps"])  # photons across a cut in mid range
            assert np.array_equal(g.em_host_state(p), gam)
        out.append((x, gam))
        g.close()
    dx = _norm_dev(out[0][0], out[1][0])
    dg = np.linalg.norm(out[0][1] - out[1][1]) / np.linalg.norm(out[1][1])
    print(f"K={K}: nuclei {dx:.2e}, photons {dg:.2e}")
    assert dx <= TOL and dg <= TOL


@pytest.mark.parametrize("K,two", [(1, True), (3, False), (8, True), (13, True), (40, False),
                                   (70, True)])
def test_adjoint_march_equals_the_transposed_stages(K, two):
    """The adjoint sweep by marches against the per-step kernels, more than one
    checkpoint chunk, ragged columns."""
    import torch

    run = workloads.nuclear_run()
    out = []
    for team in (True, False):
        g = _solver(run, 0.07, K, 7, team, np.linspace(0.6, 1.4, K) if two else None)
        p = g.prepare(1e-3, with_adjoint=True)
        assert ((p.get("team_adjoint") is not None) == team)
        lam = torch.randn(tuple(p["x"].shape), dtype=torch.float64,
                          generator=torch.Generator().manual_seed(2)).to(p["x"].device)
        res = []
        for _ in range(2):
            g.forward_checkpointed(p)
            ab = g.adjoint_sweep(p, lam)
            res.append({k: ab[k].clone() for k in ("lam", "gsrc0", "gsrc1", "gdot")})
        assert all(torch.equal(res[0][k], res[1][k]) for k in res[0])
        out.append(res[0])
        g.close()
    for k in ("lam", "gsrc0", "gsrc1") + (("gdot",) if two else ()):
        d = _norm_dev(out[0][k], out[1][k])
        print(f"K={K} {k}: {d:.2e}")
        assert d <= TOL, k


def test_displaced_tables_outlive_their_use_on_another_stream():
    """Two plans on two streams share a layout's tables.  Displaced and dropped while
    the second stream still marches, their memory is not given to new tensors of the
    stream that made them."""
    import torch

    run = workloads.nuclear_run()
    K = 65  # no other test's plan
    g = _solver(run, 2.0, K, 11, True)
    p = g.prepare(1e-3)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        g2 = _solver(run, 2.0, K, 11, True)
        p2 = g2.prepare(1e-3)
    shared = ("rows", "mothers", "lds_voff", "dense_ent")
    ptrs = {n: p2["team"]["bufs"][n].data_ptr() for n in shared}
    sizes = {n: p2["team"]["bufs"][n].numel() for n in shared}
    assert all(p["team"]["bufs"][n].data_ptr() == q for n, q in ptrs.items())
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        want = g2.execute(p2).clone()
        torch.cuda.synchronize()
        x = g2.execute(p2)  # about 70 ms on the side stream
    for lay in g._device_cache().layouts.values():
        for key in [k for k in lay.get("team", {}) if k[0] == K]:
            del lay["team"][key]
    g.close()
    g2.close()
    del p, p2
    new = [torch.empty(n, dtype=torch.int32, device=x.device) for n in sizes.values() for _ in range(8)]
    assert not side.query(), "the march ended too early for this test"
    assert not {t.data_ptr() for t in new} & set(ptrs.values())
    torch.cuda.synchronize()
    assert torch.equal(x, want)


@pytest.mark.parametrize("K", [1, 2, 40])
def test_stencil_coefficients_outside_the_grid_are_not_used(K):
    """An operator whose table holds numbers there: as the stage kernels, the march
    gives what it gives for zeros."""
    import torch

    g = _solver(workloads.nuclear_run(), 0.02, K, 12, True)
    p = g.prepare(1e-3)
    want = g.execute(p).clone()
    t = p["bufs"]["dcoef"].view(64, 7)
    bins = torch.arange(64, device=t.device)[:, None] + torch.arange(-3, 4, device=t.device)[None, :]
    outside = (bins < 0) | (bins > 63)
    assert int(outside.sum()) == 12 and not bool(t[outside].any())
    t[outside] = 3.0
    assert torch.equal(g.execute(p), want)


@pytest.mark.parametrize("K", [1, 9, 40])
def test_injection_without_sources_adds_nothing(K):
    """The flag set and no sources (nsrc 0): no coefficient is read, and the steps are
    those without the flag, as in the stage kernels."""
    import torch

    from prince_amd import _lib

    g = _solver(workloads.nuclear_run(), 0.02, K, 13, True)
    p = g.prepare(1e-3)
    x0 = torch.rand(tuple(p["x"].shape), dtype=torch.float64,
                    generator=torch.Generator().manual_seed(1)).to(p["x"].device)
    g.fold_windows(p)
    out = []
    for nsrc, flags in ((0, p["op"].flags), (p["op"].nsrc, p["op"].flags & ~_lib.PRH_F_INJECTION)):
        p["op"].nsrc, p["op"].flags = nsrc, flags
        p["x"].copy_(x0)
        g._launch_steps(p, 0, p["nsteps"])
        out.append(p["x"].clone())
    assert torch.equal(*out) and not torch.equal(out[0], x0)
