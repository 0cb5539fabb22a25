"""Team-march plans (``solvers/team.py``) replayed in numpy on the host-built
layout: every row once, every index inside its table, the values in LDS slots
reproduce the off-diagonal product and the diagonal."""

import numpy as np
import pytest

from prince_amd import workloads
from prince_amd.solvers import team
from prince_amd.solvers.layout import build_block_layout


@pytest.fixture(scope="module")
def layouts():
    out = {}
    for name, run in (("proton", workloads.proton_run()), ("nuclear", workloads.nuclear_run())):
        M = run.int_rates.coupling_mat.tocsr()
        m0 = run.int_rates._batch_matrix @ run.int_rates.photon_vector(1.0)
        out[name] = (build_block_layout(M.indptr, M.indices, m0, run.spec_man.nspec, 64), M, m0)
    return out


def _shift(x, o):
    y = np.zeros_like(x)
    y[: 64 - o] = x[o:]
    return y


@pytest.mark.parametrize("em", [False, True])
@pytest.mark.parametrize("name,K,fields,size", [
    ("proton", 1, 1, None), ("proton", 9, 2, None), ("nuclear", 1, 1, None),
    ("nuclear", 7, 2, None), ("nuclear", 37, 1, 64), ("nuclear", 64, 1, None),
    ("nuclear", 64, 1, 256), ("nuclear", 300, 2, 128), ("nuclear", 512, 1, None)])
def test_plan_reproduces_the_operator(layouts, name, K, fields, size, em):
    lay, M, m0 = layouts[name]
    nspec, n = lay.nspec, lay.n
    blocks = lay.blocks.copy()
    blocks[:, 3] += n
    vals = np.concatenate([np.where(lay.sel < 0, 0.0, m0[np.maximum(lay.sel, 0)])[lay.zslots:],
                           np.where(lay.sel < 0, 0.0, m0[np.maximum(lay.sel, 0)])[: lay.zslots]])
    p = team.build_team(blocks, lay.brow_ptr, nspec, 64, 0, K, fields, em=em, size=size)
    assert p is not None and p.nteam * p.size <= team.CUS
    assert p.lds_bytes(fields) <= team.LDS_BYTES
    assert p.lds_ptr.size == p.size + 1 and p.wave_ptr.size == p.size * team.WAVES + 1
    assert np.all((p.lds_voff[:, 0] >= 0) & (p.lds_voff[:, 0] + 64 <= vals.size))
    x = np.random.default_rng(3).standard_normal((nspec, 64))
    got = np.full((nspec, 64), np.nan)
    diag = np.full((nspec, 64), np.nan)
    part = np.zeros((max(1, p.nparts), 64))
    tail = set(p.fin[:, 0].tolist())
    assert p.fin.shape[0] == len(tail) and set(p.dense_rows) <= tail
    for rank in range(p.size):
        lds = []
        for v, sh in p.lds_voff[p.lds_ptr[rank]:p.lds_ptr[rank + 1]]:
            assert sh == 0 or rank < p.ndwg
            lds.append(np.concatenate([np.zeros(sh), vals[v:v + 64 - sh]]))
        mult = 2 if p.ndwg <= rank < p.ndwg + p.nfwg else 1
        assert mult * len(lds) <= p.lds_slots
        if rank < p.ndwg:
            e0, e1 = p.dense_ptr[rank * p.dgroups], p.dense_ptr[(rank + 1) * p.dgroups]
            assert np.all(np.diff(p.dense_ptr) <= 64) and e1 >= e0
            for mo, s0, b0, s1, b1 in p.dense_ent[e0:e1]:
                assert mo not in tail
                for r, (s, b) in enumerate(((s0, b0), (s1, b1))):
                    for i in range(b >> 8):  # the value in the mother's bins
                        part[(3 if em else 2) * rank + r] += _shift(lds[s + i] * x[mo], (b & 255) + i)
        if rank < p.ndwg + p.nfwg:
            assert p.wave_ptr[rank * team.WAVES] == p.wave_ptr[(rank + 1) * team.WAVES]
            continue
        wp = p.wave_ptr[rank * team.WAVES:(rank + 1) * team.WAVES + 1]
        if p.pair_rows:  # two waves share each task
            for w in range(0, team.WAVES, 2):
                assert np.array_equal(p.rows[wp[w]:wp[w + 1]], p.rows[wp[w + 1]:wp[w + 2]])
            waves = range(0, team.WAVES, 2)
        else:
            waves = range(team.WAVES)
        for t in (t for w in waves for t in range(wp[w], wp[w + 1])):
            a, b, n2, na, nb, ga, gb, pa, pb, m = p.rows[t]
            ent = p.mothers[m:m + n2 + na + nb]
            assert n2 + na + nb <= 64 and not tail.intersection(ent[:, 0].tolist())
            assert p.pair_rows or b < 0
            both, ea, eb = ent[:n2], ent[n2:n2 + na], ent[n2 + na:]
            for da, dg, ps, mine, at in ((a, ga, pa, ea, 0), (b, gb, pb, eb, 1)):
                if da < 0:
                    assert at == 1 and n2 == nb == 0
                    continue
                assert np.isnan(got[da, 0]) and (ps >= 0) == (da in tail)
                s = sum((lds[q[1] + at] * x[q[0]] for q in both), np.zeros(64))
                s = sum((lds[q[1]] * x[q[0]] for q in mine), s)
                if ps >= 0:
                    part[ps] = s
                else:
                    got[da], diag[da] = s, lds[dg]
    if em and p.ndwg:  # every heavy row has a weight in exactly one dense entry
        heavy = sorted(set(range(nspec)) - tail)
        assert sorted(p.dense_ent[:, 0].tolist()) == heavy
    if p.nfwg:  # every finishing workgroup holds the same slots
        r = p.ndwg
        fl = [vals[v:v + 64] for v, _ in p.lds_voff[p.lds_ptr[r]:p.lds_ptr[r + 1]]]
        for k in range(r, r + p.nfwg):
            assert np.array_equal(p.lds_voff[p.lds_ptr[k]:p.lds_ptr[k + 1]],
                                  p.lds_voff[p.lds_ptr[r]:p.lds_ptr[r + 1]])
        for da, slot, p0, pstep, pn, b0, nb, _ in p.fin:
            assert np.isnan(got[da, 0]) and (pn == 0 or p0 + pstep * (pn - 1) < p.nparts)
            got[da] = sum((part[p0 + g * pstep] for g in range(pn)), np.zeros(64))
            diag[da] = fl[slot]
            for mo, s, ol, ns in p.fin_blk[b0:b0 + nb]:
                assert mo in tail
                for i in range(ns):
                    got[da] = got[da] + fl[s + i] * _shift(x[mo], ol + i)
    full = M.copy()
    full.data = m0.copy()
    d = full.diagonal()
    want = (full @ x.ravel() - d * x.ravel()).reshape(nspec, 64)
    # sums of up to 2500 products in another order: 2500 eps of the largest term
    assert np.allclose(got, want, rtol=1e-12, atol=1e-12 * np.abs(want).max())
    assert np.array_equal(diag.ravel(), d)


def test_column_tilings_cover_the_columns():
    for nc in range(1, 140):
        kd, g = team.dense_tiling(nc)
        assert kd in (1, 2) and team.WAVES % g == 0
        assert g == 1 or (g >= 2 and kd == 1 and team.WAVES // g * 2 >= nc)
        pairs, kp = team.row_tiling(nc)
        assert kp in (1, 2) and (pairs or (nc <= 2 and kp == 1))


def test_operators_outside_the_march_are_refused():
    diag = np.array([[0, 0, 1, 0]])
    ptr = np.array([0, 1])
    assert team.build_team(diag, ptr, 1, 64, 0, 1) is not None
    assert team.build_team(diag, ptr, 1, 32, 0, 1) is None  # other bin counts
    assert team.build_team([[0, -3, 4, 0]], ptr, 1, 64, 0, 1) is None  # left bands
    assert team.build_team([[0, 0, 9, 0]], ptr, 1, 64, 0, 1) is None  # wide bands
    three = np.tile([0, 0, 8, 0], (3, 1))
    assert team.build_team(three, np.arange(4), 3, 64, 0, 1) is None  # three band rows
    chain = np.array([[1, 0, 8, 0]] + [[i - 1, 0, 1, 64 * i] for i in range(1, 40)])
    assert team.build_team(chain, np.arange(41), 40, 64, 0, 1) is None  # every row reads the tail
    assert team.build_team(diag, ptr, 1, 64, 0, 5_000_000) is None  # state beyond 2 GiB
    assert team.build_team(diag, ptr, 1, 64, 0, 64, nsrc=128) is not None
    assert team.build_team(diag, ptr, 1, 64, 0, 64, nsrc=129) is None  # coefficients per team


@pytest.mark.parametrize("name,K,fields,size", [
    ("proton", 3, 2, None), ("nuclear", 1, 1, None), ("nuclear", 64, 2, None),
    ("nuclear", 37, 2, 128), ("nuclear", 300, 1, None)])
def test_adjoint_plan_reproduces_the_transposed_operator(layouts, name, K, fields, size):
    from prince_amd.solvers.layout import transposed_layout

    lay, M, m0 = layouts[name]
    nspec, n = lay.nspec, lay.n
    tr = transposed_layout(M.indptr, M.indices, m0, nspec, 64)
    blocks = tr.blocks.copy()
    blocks[:, 3] += n
    pick = np.where(tr.sel < 0, 0.0, m0[np.maximum(tr.sel, 0)])
    vals = np.concatenate([pick[tr.zslots:], pick[:tr.zslots]])
    p = team.build_adjoint_team(blocks, tr.brow_ptr, nspec, 64, 0, K, fields, size=size)
    nc = -(-K // p.nteam)
    assert np.all((p.lds_voff[:, 0] >= 0) & (p.lds_voff[:, 0] + 64 <= vals.size))
    x = np.random.default_rng(4).standard_normal((nspec, 64))
    got = {}
    for rank in range(p.size):
        lds = [vals[v:v + 64] for v, _ in p.lds_voff[p.lds_ptr[rank]:p.lds_ptr[rank + 1]]]
        assert len(lds) <= p.lds_slots
        for t in range(p.wave_ptr[rank * 16], p.wave_ptr[(rank + 1) * 16]):
            r, nd, nb, head, cg, ncg, first = (int(v) for v in p.rows[t][:7])
            assert nd + nb <= 64 and np.array_equal(lds[head], vals[64 * r:64 * r + 64])
            y = np.zeros(64)
            for e, (mo, sl, ol, ns) in enumerate(p.mothers[first:first + nd + nb].tolist()):
                assert (ns == 1 and ol == 0) if e < nd else (ns <= 8 and ol + ns <= 1)
                for i in range(ns):
                    sh = np.zeros(64)
                    o = -(ol + i)
                    sh[o:] = x[mo][:64 - o]
                    y += lds[sl + i] * sh
            got.setdefault(r, []).append((cg, ncg, y))
    full = M.copy()
    full.data = m0.copy()
    want = (full.T @ x.ravel() - full.diagonal() * x.ravel()).reshape(nspec, 64)
    for r in range(nspec):  # every pair of columns by exactly one wave
        pairs = sorted(q for cg, ncg, _ in got[r] for q in range(cg, -(-nc // 2), ncg))
        assert pairs == list(range(-(-nc // 2)))
        assert np.allclose(got[r][0][2], want[r], rtol=1e-12, atol=1e-12 * np.abs(want).max())


def test_kept_plans_are_shared_by_threads():
    """Threads that prepare solves on one run at once: each gets the plan of its own
    size while the others' displace it."""
    import sys
    import threading

    lay, wrong = {}, []

    def work(seed):
        rng = np.random.default_rng(seed)
        try:
            for k in rng.integers(0, 12, size=4000).tolist():
                if team.kept(lay, k, lambda: ("plan", k), 3) != ("plan", k):
                    wrong.append(k)
        except Exception as e:  # noqa: BLE001
            wrong.append(repr(e))

    old = sys.getswitchinterval()
    sys.setswitchinterval(1e-6)
    try:
        threads = [threading.Thread(target=work, args=(i,)) for i in range(8)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    finally:
        sys.setswitchinterval(old)
    assert not wrong and 0 < len(lay["team"]) <= 3
