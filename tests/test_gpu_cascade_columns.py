"""GPU: the column blocks of prh_cascade_transfer against the host builder where
their work differs: iterations cut off by the cap, matrices that are not upper
triangular (all tiles), a column whose energy rises above tol again after every
block had converged (the windows' common last iterations)."""

import copy

import numpy as np
import pytest

from prince_amd import workloads
from prince_amd.model import cascade as C
from prince_amd.solvers.cascade_device import DeviceCascade

pytestmark = pytest.mark.gpu

# about 40 iterations of sums over at most 144 terms in FP64: 40 * 144 * 1.1e-16 = 6e-13
TOL = 1e-11


@pytest.mark.parametrize("what, cap, tol", [
    ("plain", C.MAX_SCATTER, C.CASCADE_TOL),
    ("plain", 1, C.CASCADE_TOL),
    ("plain", 3, C.CASCADE_TOL),
    ("no weight", C.MAX_SCATTER, C.CASCADE_TOL),
    ("lower", C.MAX_SCATTER, C.CASCADE_TOL),
    ("rise", C.MAX_SCATTER, 1.1),
])
def test_column_blocks_match_host(what, cap, tol):
    import torch

    run = workloads.proton_em_run()
    ck = copy.copy(C.cascade_kernels(run.em_grid.grid, run.cr_grid.grid))
    if what in ("no weight", "lower"):  # pairs above the photon's energy: below the diagonal
        ck.A_pair = ck.A_pair.copy()
        if what == "no weight":  # no photon pairs at the lower bin: stays triangular
            ck.A_pair[100, 40] = ck.A_pair[:, 100].max(axis=0)
        else:
            ck.A_pair[130, 100] = ck.A_pair[:, 110].max(axis=0)
    if what == "rise":  # every degraded electron in the upper of its two bins
        ck._cic_f = np.zeros_like(ck._cic_f)
    dc = DeviceCascade(ck, torch.device("cuda", 0))
    dc.cs.max_scatter, dc.cs.tol = cap, tol
    zs = np.array([1.2, 3.0])
    tg, te, _, iters = (t.cpu().numpy() for t in dc.build(zs, run.photon_field, 1e-3))
    for w, z in enumerate(zs):
        Tg, Te, it = ck.transfer_one(z, run.photon_field, 1e-3, max_scatter=cap, tol=tol)
        assert iters[w] == it
        for got, ref in ((tg[w], Tg), (te[w], Te)):
            assert np.abs(got - ref).max() <= TOL * np.abs(ref).max(), (w, z)
        if what == "lower":
            low, lowref = np.tril(tg[w], -16), np.tril(Tg, -16)
            assert lowref.max() > 0.0
            assert np.abs(low - lowref).max() <= TOL * lowref.max()
