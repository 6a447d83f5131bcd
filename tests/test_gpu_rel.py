"""The relativistic kernels of a frequency batch where their split and their
ladder cells can go wrong: batch sizes on both sides of each split, as many Gamma
rows as a wavefront takes at once and more, the smallest and the largest
principal-value windows, odd grids, and (Gamma, pparbar) tables whose rows are not
the same grid (a row's ladder then leaves the cells around its resonance).

Bar: 1e-11 of the largest |chi| of the species (tests/test_gpu_disp.py), or ten
times the oracle's own jump under a 1e-13 relative change of omega where that is
larger (a ladder end on a cell boundary)."""
import dataclasses

import numpy as np
import pytest

import cases
from alps_amd.plasma import juttner_plasma
from oracle import Oracle

pytestmark = pytest.mark.gpu

TOL = 1e-11
OMS = [0.5113 + 0.0511j, 0.5113 - 0.0511j, 0.3127 - 0.0021j, 0.1217 + 0.3j, 0.8019 + 0.0j,
       1.5131 - 0.3j]


def _oracle(p, kperp, kpar, oms):
    O = Oracle(p)
    nmax = O.set_k(kperp, kpar)
    out = []
    for om in oms:
        _, chi, low, _ = O.disp(om, want_tensors=True)
        _, chi_p, low_p, _ = O.disp(om * (1.0 + 1e-13), want_tensors=True)
        out.append((chi, low, np.abs(chi_p - chi), np.abs(low_p - low)))
    return nmax, out


def _check(p, kperp, kpar, oms, sizes=(None,)):
    from alps_amd.engine import Engine
    nmax, ref = _oracle(p, kperp, kpar, oms)
    E = Engine(p)
    assert E.set_k(kperp, kpar) == nmax
    for n in sizes:
        om = np.resize(np.array(oms), n or len(oms))
        _, chi, low, _ = E.disp_batch(om, want_tensors=True)
        for k in list(range(min(len(om), len(oms)))) + [len(om) - 1]:
            c, l, jc, jl = ref[k % len(oms)]
            for s in range(p.nspec):
                for g, o, j in ((chi[k, s], c[s], jc[s]), (low[k, s], l[s], jl[s])):
                    sc = max(np.max(np.abs(o)), 1e-300)
                    assert np.all(np.isfinite(g))
                    tol = max(TOL, 10.0 * np.max(j) / sc)
                    assert np.max(np.abs(g - o)) / sc <= tol, (n, k, om[k], s)
    E.close()


def test_batch_sizes_of_every_split():
    _check(cases.rel_mixed(), 0.3, 0.3, OMS, sizes=(1, 6, 64, 65, 256, 257))


@pytest.mark.parametrize("pos,npparbar", [(1, 203), (16, 901)])
def test_window_sizes(pos, npparbar):
    p = dataclasses.replace(cases.rel_pair(nperp=12, npar=41, ngamma=21, npparbar=npparbar),
                            positions_principal=pos)
    _check(p, 0.31, 0.29, OMS)


@pytest.mark.parametrize("ngamma,pos,sizes", [
    (100, 3, (256, 257, 300)), (200, 3, (64, 65, 256, 257)), (400, 3, (1, 64)),
    (100, 1, (300,)), (100, 2, (300,)), (150, 4, (300,)), (100, 5, (300,)),
    (100, 6, (1, 65, 257)), (150, 7, (1, 257)), (100, 10, (1, 65, 300))])
def test_many_gamma_rows(ngamma, pos, sizes):
    """All 32 Gamma rows that a wavefront of k_rel_res decides at once, and a second
    32 of them (200 rows at 257 omegas), for windows of fewer and of more cells than
    it has lanes.  The omegas' n = 0 resonances lie inside the cone on every row
    from the first few on."""
    p = juttner_plasma(ms=[1.0, 1.0], qs=[1.0, -1.0], ns=[1.0, 1.0], taus=[1.0, 1.0], beta=1.0,
                       vA=1.0, nperp=12, npar=24 if pos < 10 else 41, maxP=5.0, ngamma=ngamma,
                       npparbar=400 if pos > 5 else 200, analytic_rel=True,
                       positions_principal=pos, n_resonance_interval=100, Tlim=0.01,
                       Bessel_zero=1e-45)
    _check(p, 0.3, 0.3, [0.1217 + 0.03j, 0.2113 + 0.0011j, 0.1531 - 0.004j], sizes=sizes)


def test_far_omegas():
    """omegas whose |den|^2 of four harmonics have no product in double precision
    (beyond 3e38), and one on the other side: D is finite up to 1e50"""
    _check(cases.rel_pair(), 0.3, 0.3, [1e30 + 1e29j, 1e39 + 2e38j, 1e40 + 1e39j, 1e45 - 1e44j],
           sizes=(4, 300))


def test_rows_on_grids_of_their_own():
    """Row ig of pparbar_rel shifted by up to five steps: the ladder of a row,
    laid out from rows 1 and 2, crosses cells away from its resonance's."""
    p = cases.rel_pair(nperp=12, npar=24, ngamma=20, npparbar=200)
    pb, f0, df = p.pparbar_rel.copy(), p.f0_rel.copy(), p.df0_rel.copy()
    d = pb[0, 2, 2] - pb[0, 2, 1]
    for ig in range(3, pb.shape[1]):
        pb[:, ig] += d * (0.37 + 5.0 * np.sin(1.7 * ig))
    out = (p.gamma_rel ** 2 - 1.0) < pb ** 2
    f0[out] = -1.0
    df[out] = 0.0
    _check(dataclasses.replace(p, pparbar_rel=pb, f0_rel=f0, df0_rel=df), 0.3, 0.3,
           OMS[:5])
