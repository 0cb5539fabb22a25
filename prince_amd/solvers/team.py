"""Plan of the team march (``prh_team_march``): which workgroup of a team owns
which species rows, and where their coupling values sit in its LDS.

A team is ``size`` workgroups of 16 waves (one per CU), ``nteam`` teams fill the
chip and each marches its own share of the right-hand sides.  Heavy rows
(diagonal blocks only) go one per wave, or from 3 right-hand sides per team on as
pairs of consecutive rows, read with one walk over their mothers by two waves that
share the right-hand sides.  The tail rows -- the dense rows (at most
two: band blocks or more than ``ROW_MAX`` blocks) and every row that reads a tail
row -- run one stage behind them: ``ndwg`` workgroups sum the dense rows over the
heavy mothers, each taking a contiguous range of mothers for both rows, the other
tail rows' sums over heavy mothers run among the heavy rows, and ``nfwg``
workgroups finish the tail rows.  Pure numpy.
"""

from __future__ import annotations

import threading
from dataclasses import dataclass

import numpy as np

WAVES = 16
CUS = 256
#: LDS bytes a workgroup may use (160 KB per CU less the kernel's static words)
LDS_BYTES = 160 * 1024 - 64
CONST_SLOTS = 9
ROW_MAX = 32
DENSE_MAX = 2
BAND_MAX = 8
TAIL_MAX = 32
SYNC_BYTES = 18688


# Right-hand sides up to which a march beats the stage kernels, by species rows: (rows
# from, K below 256, K from 256 on, where the stage kernels take 8 right-hand sides per
# wave).  A march has at most 8 teams; few rows leave most of a team's workgroups idle,
# so its columns queue up where the stage kernels fill the chip.  Stage kernels over
# march, time per step, at K inside a line | beyond it:
#   one field   1 row     255 1.22, 448 1.05 | 512 0.94, 4096 0.15
#               2         192 1.10, 256 - 320 1.21 - 1.04 | 224 0.92, 384 0.92
#               4 - 41    128 0.99 - 1.33 | 192 0.67 - 1.06, 256 0.74 - 1.04, 512 0.54
#               53 - 77   128 1.21 - 1.47, 288 1.06 - 1.20 | 160 0.85 - 1.04, 384 0.87 - 1.01
#               89, 113   384 1.01, 1.11 | 512 0.84
#               137       448 1.05 | 512 0.95
#               209       768 1.04 | 896 0.97
#               257, 305  512 1.32, 1.18 | 640 1.11, 0.93; 1024 1.00, 0.95
#   two fields  1 row     160 1.01, 512 1.06 | 192 0.98
#               2 - 41    64 1.16 - 1.40 | 80 0.77 - 0.95, 256 0.86 - 1.00
#               53 - 77   96 0.99 - 1.11, 256 1.15 - 1.32 | 160 0.73, 384 0.85 - 0.92
#               89, 113   320 1.10, 1.25 | 384 0.93, 1.06
#               137, 173  384 1.11, 1.30; 448 1.21 | 512 0.95, 1.15
#               209       768 1.21
#               257, 305  384 0.93, 1.04 | 512 0.85, 0.97
# With the EM cascade as one field (305 rows 512 1.20 | 640 0.99; 7 rows 128 1.24 | 512 0.63).
MARCH_PAYS = {
    1: ((1, 255, 448), (2, 192, 320), (3, 128, 0), (48, 128, 288), (85, 255, 384), (120, 255, 448),
        (200, 255, 768), (250, 255, 512)),
    2: ((1, 160, 512), (2, 64, 0), (48, 96, 288), (85, 255, 320), (120, 255, 448), (200, 255, 768),
        (250, 255, 384)),
}
# A gradient's forward stages (16 waves, no row pairs) lose to the march for longer: one
# field, 305 rows, 1024 1.25.
GRADIENT_ROWS, GRADIENT_K = 200, 2048
# The adjoint march, by the time of a sweep:
#   one field   1, 2 rows  512 1.13, 1.00 | 768 0.85;  7 512 1.11;  17 2048 1.03;  53 - 305 1.09 - 1.40
#   two fields  1 row      128 1.00 | 160 0.95;  2 64 1.12 | 80 0.92;  7 80 1.07 | 128 0.93
#               17         255 1.04, 448 1.12;  35 128 1.00 | 192 0.88;  53 80 1.14 | 128 0.92
#               89, 137    128 1.07, 1.06 | 255 0.91, 0.96
#               209, 305   128 0.98, 1.01 | 192 0.89, 0.96
ADJOINT_PAYS = {
    1: ((1, 255, 512), (8, 255, 2048)),
    2: ((1, 128, 0), (2, 64, 0), (3, 80, 0), (8, 255, 448), (29, 128, 0), (48, 80, 0), (85, 128, 0)),
}


def _within(lines, nspec, K):
    _, below, above = [ln for ln in lines if ln[0] <= nspec][-1]
    return K <= (below if K < 256 else above)


def march_pays(nspec, K, fields, gradient=False):
    """Whether the march beats the stage kernels for K right-hand sides."""
    if gradient and fields == 1 and nspec >= GRADIENT_ROWS:
        return K <= GRADIENT_K
    return _within(MARCH_PAYS[fields], nspec, K)


def adjoint_march_pays(nspec, K, fields):
    """The same for the adjoint sweep."""
    return _within(ADJOINT_PAYS[fields], nspec, K)


_KEPT_LOCK = threading.Lock()


def kept(lay, key, make, most):
    """``make()`` of a key, kept with the layout ``lay``; at most ``most`` of them, the
    oldest goes first.  Solvers of several threads share a layout."""
    with _KEPT_LOCK:
        value = lay.setdefault("team", {}).get(key)
    if value is None:
        value = make()
        with _KEPT_LOCK:
            plans = lay["team"]
            value = plans.setdefault(key, value)
            while len(plans) > most:
                plans.pop(next(k for k in plans if k != key))
    return value


@dataclass
class TeamPlan:
    nteam: int
    size: int
    kp: int
    kd: int
    dgroups: int
    ndwg: int
    nfwg: int
    pair_rows: bool
    nparts: int
    dense_rows: list
    lds_slots: int
    red_slots: int
    coef_slots: int
    lds_ptr: np.ndarray
    lds_voff: np.ndarray
    wave_ptr: np.ndarray
    rows: np.ndarray
    mothers: np.ndarray
    dense_ptr: np.ndarray
    dense_ent: np.ndarray
    fin: np.ndarray
    fin_blk: np.ndarray

    def lds_bytes(self, fields):
        return 512 * (CONST_SLOTS + 2 * fields + 2 * self.coef_slots + self.red_slots + fields * self.lds_slots)


def dense_tiling(nc):
    """(kd, dgroups) of the dense-row workgroups for ``nc`` columns per team: the
    16 waves are column groups of ``kd`` pairs of columns times mother groups;
    mother groups only while one pass of single pairs covers the columns."""
    if nc <= 16:
        pairs = 1
        while 2 * pairs < nc:
            pairs *= 2
        return 1, WAVES // pairs
    return (1 if nc <= 32 else 2), 1


def row_tiling(nc):
    """(row pairs or not, pairs of right-hand sides per pass of a wave)."""
    return nc > 2, 1 if nc <= 4 else 2


def _cut(cost, parts):
    """Cut a cost list into ``parts`` contiguous ranges of similar cost (bounds)."""
    c = np.concatenate([[0.0], np.cumsum(cost)])
    at = np.searchsorted(c, c[-1] * np.arange(1, parts) / parts, side="left")
    return np.concatenate([[0], np.minimum(at, len(cost)), [len(cost)]]).astype(np.int64)


def tail_rows(blocks, ptr, nspec):
    """(dense rows, tail rows): the tail is the smallest set that holds the dense
    rows and every row that reads a row of the set."""
    dense = []
    for da in range(nspec):
        b = blocks[ptr[da]:ptr[da + 1]]
        if len(b) > ROW_MAX or not np.all((b[:, 1] == 0) & (b[:, 2] == 1)):
            dense.append(da)
    tail = set(dense)
    grown = bool(tail)
    while grown:
        grown = False
        for da in range(nspec):
            if da not in tail and tail.intersection(blocks[ptr[da]:ptr[da + 1], 0].tolist()):
                tail.add(da)
                grown = True
    return dense, sorted(tail)


def build_team(blocks, brow_ptr, nspec, d, diag_off, K, fields=1, nsrc=1, em=False, size=None):
    """Team plan of an operator for K right-hand sides, or None when its rows do
    not fit the march (d != 64, more than two dense rows, bands left of the
    diagonal or wider than 8, a long tail, values beyond the LDS, more source
    coefficients per team than threads).  ``em``: the march also forms the
    Bethe-Heitler sums (every heavy row gets a dense entry)."""
    if d != 64 or nspec < 1 or nspec * K * 512 > 0x7FFFFFFF:
        return None
    blocks = np.asarray(blocks, dtype=np.int64).reshape(-1, 4)
    ptr = np.asarray(brow_ptr, dtype=np.int64)
    dense, tail = tail_rows(blocks, ptr, nspec)
    if len(dense) > DENSE_MAX or len(tail) > TAIL_MAX or (em and not tail):
        return None
    # the second dense row is the one of single diagonals
    dense.sort(key=lambda da: -int(blocks[ptr[da]:ptr[da + 1], 2].max()))
    if len(dense) == 2:
        b = blocks[ptr[dense[1]]:ptr[dense[1] + 1]]
        if np.any(b[:, 2] > 1) or np.any(b[:, 1] != 0):
            return None
    for da in dense:
        b = blocks[ptr[da]:ptr[da + 1]]
        if np.any(b[:, 1] < 0) or np.any(b[:, 1] + b[:, 2] > BAND_MAX):
            return None
    sizes = [1] if len(tail) == nspec else [size] if size is not None else [32, 64, 128, 256]
    for s in sizes:
        plan = _build(blocks, ptr, nspec, dense, tail, diag_off, K, fields, nsrc, em, s)
        if plan is not None:
            return plan
    return None


def _build(blocks, ptr, nspec, dense, tail, diag_off, K, fields, nsrc, em, size):
    nteam = min(8, CUS // size)
    nc = -(-K // nteam)
    kd, dgroups = dense_tiling(nc)
    pair_rows, kp = row_tiling(nc)
    if nsrc * nc > 64 * WAVES:
        return None
    coef = -(-nsrc * nc // 64)
    tset = set(tail)
    # dense entries: one per heavy mother, both rows' blocks
    ent = {}
    for r, da in enumerate(dense):
        for v in range(int(ptr[da]), int(ptr[da + 1])):
            mo, ol, ns, vo = (int(q) for q in blocks[v])
            if mo not in tset:
                ent.setdefault(mo, [[0, 0, 0], [0, 0, 0]])[r] = [ol, ns, vo]
    if em:
        for da in range(nspec):
            if da not in tset:
                ent.setdefault(da, [[0, 0, 0], [0, 0, 0]])
    mothers = sorted(ent)
    eslots = np.array([sum(q[1] for q in ent[m]) for m in mothers], dtype=np.int64)
    nsum = DENSE_MAX + int(em)
    red = WAVES * nsum * 2 if (mothers and dgroups > 1) else 0
    budget = (LDS_BYTES // 512 - CONST_SLOTS - 2 * fields - 2 * coef - red) // fields
    ndwg = 0
    if mothers:
        # the least number of workgroups whose LDS holds the dense values
        ndwg = max(1, -(-int(eslots.sum()) // max(1, budget)))
        while ndwg < size and max(eslots[a:b].sum() for a, b in zip(*_bounds(eslots, ndwg))) > budget:
            ndwg += 1
    heavy = [da for da in range(nspec) if da not in tset]
    # tail rows that are not dense sum their heavy mothers among the heavy rows
    light = [da for da in tail if da not in dense]
    nfwg = 0 if not tail else 1 if size == 1 or len(tail) * nc <= WAVES else 2
    nrow_wg = size - ndwg - nfwg
    if nrow_wg < (1 if heavy else 0):
        return None
    lds_ptr, lds_voff = [0], []
    dptr, dent = [0], []
    wave_ptr, rows, mlist = [0], [], []
    if ndwg:
        for a, b in zip(*_bounds(eslots, ndwg)):
            voff = []
            slot = {}
            for e in range(a, b):
                q = []
                for ol, ns, vo in ent[mothers[e]]:
                    q += [len(voff) if ns else 0, ol | ns << 8]
                    # diagonal o sits o bins up, in line with the mother's bins
                    voff += [(vo + 64 * s, ol + s) for s in range(ns)]
                slot[e] = q
            for g in range(dgroups):  # mother groups: contiguous, similar counts
                lo, hi = a + (b - a) * g // dgroups, a + (b - a) * (g + 1) // dgroups
                if hi - lo > 64:
                    return None
                dent += [[mothers[e]] + slot[e] for e in range(lo, hi)]
                dptr.append(len(dent))
            lds_voff += voff
            lds_ptr.append(len(lds_voff))
            wave_ptr += [0] * WAVES
    # finishing workgroups: every tail row's diagonal and its blocks from tail mothers
    fin, fin_blk, fvoff = [], [], []
    for da in tail:
        first = len(fin_blk)
        slot = len(fvoff)
        fvoff.append((diag_off + da * 64, 0))
        for v in range(int(ptr[da]), int(ptr[da + 1])):
            mo, ol, ns, vo = (int(q) for q in blocks[v])
            if mo in tset:
                fin_blk.append([mo, len(fvoff), ol, ns])
                fvoff += [(vo + 64 * s, 0) for s in range(ns)]
        p0, pstep, pn = ((dense.index(da), nsum, ndwg) if da in dense
                         else (nsum * ndwg + light.index(da), 1, 1))
        fin.append([da, slot, p0, pstep, pn, first, len(fin_blk) - first, 0])
    for _ in range(nfwg):
        lds_voff += fvoff
        lds_ptr.append(len(lds_voff))
        wave_ptr += [0] * WAVES
    # rows over heavy mothers in species order (neighbouring rows share mothers)
    rowlist = []
    for da in sorted(light + heavy):
        b = blocks[ptr[da]:ptr[da + 1]]
        b = b[[int(m) not in tset for m in b[:, 0]]] if da in tset else b
        rowlist.append((da, b, nsum * ndwg + light.index(da) if da in tset else -1))
    per = 2 if pair_rows else 1
    lanes = WAVES // per  # tasks that run at once in a workgroup
    tasks = [rowlist[i:i + per] for i in range(0, len(rowlist), per)]
    # a mother panel loaded costs 1, a row's own state, factors and epilogue about 5
    cost = np.array([5.0 * len(t) + len(set(m for _, b, _ in t for m in b[:, 0].tolist()))
                     for t in tasks])
    if nrow_wg:
        bounds = _cut(cost, nrow_wg) if tasks else np.zeros(nrow_wg + 1, dtype=np.int64)
        if len(tasks) <= nrow_wg * lanes:  # one task at a time
            for i in range(nrow_wg):
                bounds[i + 1] = min(max(bounds[i + 1], len(tasks) - (nrow_wg - 1 - i) * lanes),
                                    bounds[i] + lanes)
        for i in range(nrow_wg):
            voff = []
            per_lane = [[] for _ in range(lanes)]
            load = [0.0] * lanes
            for t in sorted(range(bounds[i], bounds[i + 1]), key=lambda q: -cost[q]):
                w = min(range(lanes), key=lambda q: load[q])
                load[w] += cost[t]
                per_lane[w].append(t)
            for w in range(lanes):
                mine = [_row_task(tasks[t], voff, mlist, diag_off) for t in per_lane[w]]
                if any(m is None for m in mine):
                    return None
                for _ in range(per):
                    rows += mine
                    wave_ptr.append(len(rows))
            lds_voff += voff
            lds_ptr.append(len(lds_voff))
    n = np.diff(lds_ptr)
    n[ndwg:ndwg + nfwg] *= 2
    plan = TeamPlan(
        nteam=nteam, size=size, kp=kp, kd=kd, dgroups=dgroups, ndwg=ndwg,
        nfwg=nfwg, pair_rows=pair_rows, nparts=nsum * ndwg + len(light), dense_rows=list(dense),
        lds_slots=int(n.max()), red_slots=red, coef_slots=coef,
        lds_ptr=np.asarray(lds_ptr, dtype=np.int32), lds_voff=np.asarray(lds_voff, dtype=np.int32).reshape(-1, 2),
        wave_ptr=np.asarray(wave_ptr, dtype=np.int32),
        rows=np.asarray(rows, dtype=np.int32).reshape(-1, 10),
        mothers=np.asarray(mlist, dtype=np.int32).reshape(-1, 2),
        dense_ptr=np.asarray(dptr, dtype=np.int32),
        dense_ent=np.asarray(dent, dtype=np.int32).reshape(-1, 5),
        fin=np.asarray(fin, dtype=np.int32).reshape(-1, 8),
        fin_blk=np.asarray(fin_blk, dtype=np.int32).reshape(-1, 4))
    return plan if plan.lds_bytes(fields) <= LDS_BYTES else None


def _row_task(rows, voff, mlist, diag_off):
    """Task of one or two rows: their values appended to ``voff``, their mothers to
    ``mlist`` (those of both rows first)."""
    head = []
    for da, _, part in rows:
        head.append((da, len(voff), part))
        voff.append((diag_off + da * 64, 0))
    (a, ga, pa), (b, gb, pb) = (head + [(-1, 0, -1)])[:2]
    vals = [{int(m): int(v) for m, _, _, v in q.tolist()} for _, q, _ in rows]
    both = sorted(set(vals[0]) & set(vals[1])) if len(rows) == 2 else []
    first = len(mlist)
    for m in both:
        mlist.append([m, len(voff)])
        voff += [(vals[0][m], 0), (vals[1][m], 0)]
    alone = [[m for m in sorted(v) if m not in both] for v in vals] + [[]]
    for v, ms in zip(vals, alone):
        for m in ms:
            mlist.append([m, len(voff)])
            voff.append((v[m], 0))
    if len(mlist) - first > 64:
        return None
    return [a, b, len(both), len(alone[0]), len(alone[1]), ga, gb, pa, pb, first]


def _bounds(slots, parts):
    """Contiguous ranges (starts, ends) of similar slot count."""
    b = _cut(slots.astype(np.float64), parts)
    return b[:-1], b[1:]


def build_adjoint_team(blocks, brow_ptr, nspec, d, diag_off, K, fields=1, nsrc=1, size=None):
    """Team plan of the transposed operator (``prh_team_adjoint``), or None: rows of
    diagonal blocks and bands that end at or left of the diagonal, one per wave,
    the team's columns shared by as many waves per row as the workgroup has."""
    if d != 64 or nspec < 1 or nspec * K * 512 > 0x7FFFFFFF:
        return None
    blocks = np.asarray(blocks, dtype=np.int64).reshape(-1, 4)
    ptr = np.asarray(brow_ptr, dtype=np.int64)
    if np.any(blocks[:, 2] > BAND_MAX) or np.any(blocks[:, 1] + blocks[:, 2] > 1):
        return None
    if np.any(np.diff(ptr) > 64):
        return None
    for s in [1] if nspec == 1 else [size] if size is not None else [32, 64, 128, 256]:
        nteam = min(8, CUS // s)
        nc = -(-K // nteam)
        if nsrc * nc > 64 * WAVES:
            continue
        coef = -(-nsrc * nc // 64)
        budget = (LDS_BYTES // 512 - CONST_SLOTS - fields - 2 * coef) // fields
        slots = np.array([1 + int(blocks[ptr[r]:ptr[r + 1], 2].sum()) for r in range(nspec)])
        bounds = _cut(slots + 8.0, s)
        lds_ptr, voff, wave_ptr, rows, ents = [0], [], [0], [], []
        for i in range(s):
            mine = list(range(bounds[i], bounds[i + 1]))
            ncg = max(1, min(WAVES // max(1, len(mine)), -(-nc // 2)))
            base = len(voff)
            per_wave = [[] for _ in range(WAVES)]
            for q, r in enumerate(mine):
                b = blocks[ptr[r]:ptr[r + 1]]
                diag = (b[:, 2] == 1) & (b[:, 1] == 0)
                head = len(voff) - base
                voff.append((diag_off + r * 64, 0))
                first = len(ents)
                for mo, ol, ns, vo in np.concatenate([b[diag], b[~diag]]).tolist():
                    ents.append([mo, len(voff) - base, ol, ns])
                    voff += [(vo + 64 * x, 0) for x in range(ns)]
                for cg in range(ncg):
                    per_wave[(q * ncg + cg) % WAVES].append(
                        [r, int(diag.sum()), int((~diag).sum()), head, cg, ncg, first, 0, 0, 0])
            for w in per_wave:
                rows += w
                wave_ptr.append(len(rows))
            lds_ptr.append(len(voff))
        n = int(np.diff(lds_ptr).max())
        if n <= budget:
            return TeamPlan(
                nteam=nteam, size=s, kp=1, kd=1, dgroups=1, ndwg=0, nfwg=0, pair_rows=False, nparts=0,
                dense_rows=[], lds_slots=n, red_slots=0, coef_slots=coef,
                lds_ptr=np.asarray(lds_ptr, dtype=np.int32),
                lds_voff=np.asarray(voff, dtype=np.int32).reshape(-1, 2),
                wave_ptr=np.asarray(wave_ptr, dtype=np.int32),
                rows=np.asarray(rows, dtype=np.int32).reshape(-1, 10),
                mothers=np.asarray(ents, dtype=np.int32).reshape(-1, 4),
                dense_ptr=np.zeros(1, dtype=np.int32), dense_ent=np.zeros((0, 5), dtype=np.int32),
                fin=np.zeros((0, 8), dtype=np.int32), fin_blk=np.zeros((0, 4), dtype=np.int32))
    return None
