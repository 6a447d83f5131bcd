"""The Landau tables of a frequency batch where they can go wrong: batch sizes on
both sides of the rule that builds them, omegas at the tables' edges (real axis,
last tile row, one row too deep), beside the continuation's branch points, with
omegas that are NaN or have no Landau term, the most harmonics a table holds and
one more, and the n = -1, 0, 1 parts.  Each case states how many species get
tables, and most of what they cover has to come from them (alpsg_landau_work).

Bar: a tile's series is held to 2^-51 of the sums of absolute values, so 1e-11 of
the species' largest |chi| (tests/test_gpu_disp.py) leaves 2e4 for cancellation
in the sums; against the row sums of small batches, and the oracle for some."""
import dataclasses
import math

import numpy as np
import pytest

import cases
from oracle import Oracle

pytestmark = pytest.mark.gpu

TOL = 1e-11
KPERP, KPAR = 0.3, 0.41


def _tile(p, s, kpar=KPAR):
    """side of a tile and the resonant harmonics of an omega (landau_tables)"""
    pa = p.pp[s, 2, :, 1]
    d = abs(pa[2] - pa[1])
    lo = pa[1] - p.positions_principal * d
    up = max(pa[-1], pa[-2] + p.positions_principal * d)
    return (up - lo) * (1 + 1e-6) / 64, abs(kpar) * (up - lo) / abs(p.qs[s]), lo, up


def _batch(p, n, depth, seed=5):
    rng = np.random.default_rng(seed)
    om = rng.uniform(0.02, 1.9, n) - 1j * rng.uniform(0.0, depth, n)
    om[0] = 0.7 + 0.0j
    om[1] = 0.31 - 1j * depth
    om[2:6] = 0.9 + 0.2j, 0.011 - 1e-9j, -0.4 - 0.3j * depth, 1.9 - 1j * depth
    return om


def _compare(p, om, tabs, kpar=KPAR):
    from alps_amd.engine import Engine
    E = Engine(p)
    O = Oracle(p)
    assert E.set_k(KPERP, kpar) == O.set_k(KPERP, kpar)
    got, left = E.landau_work(om)
    assert got == tabs and left < 0.5 * max(tabs, 1) * len(om) * E.get_shape(len(om))[4]
    big = E.disp_batch(om, want_tensors=True)
    parts = [E.disp_batch(om[i:i + 200], want_tensors=True) for i in range(0, len(om), 200)]
    row = [np.concatenate([np.asarray(q[j]) for q in parts]) for j in range(4)]
    for s in range(p.nspec):
        for j in (1, 2):
            g, r = np.asarray(big[j])[:, s], row[j][:, s]
            sc = np.max(np.abs(r.reshape(len(om), -1)), axis=1)
            er = np.max(np.abs((g - r).reshape(len(om), -1)), axis=1)
            ok = np.isfinite(om)
            assert np.all(er[ok] <= TOL * np.maximum(sc[ok], 1e-300)), \
                (s, j, om[ok][np.argmax(er[ok] / sc[ok])], np.max(er[ok] / sc[ok]))
    for k in list(range(8)) + [len(om) - 1]:
        _, chi, lo, _ = O.disp(om[k], want_tensors=True)
        for s in range(p.nspec):
            for g, o in ((big[1][k, s], chi[s]), (big[2][k, s], lo[s])):
                assert np.max(np.abs(g - o)) <= TOL * max(np.max(np.abs(o)), 1e-300), (k, om[k], s)
    # det alone takes the same tables
    np.testing.assert_allclose(E.disp_batch(om)[8:], np.asarray(big[0])[8:], rtol=1e-10)
    E.close()


@pytest.mark.parametrize("case,rows", [("kappa_case", 1), ("kappa_case", 7), ("kappa_case", 24),
                                       ("kappa_two_fits", 3), ("kappa_poly_mix", 2)])
def test_tile_rows(case, rows):
    """depth in tile rows of the protons, up to the tables' 24"""
    p = getattr(cases, case)()
    t, harm, _, _ = _tile(p, 0)
    n0 = max(512, math.ceil(64 * 64 * rows / harm))
    om = _batch(p, n0 + 3, (rows - 1e-3) * t * KPAR)
    _compare(p, om, 1)


@pytest.mark.parametrize("kpar,nr", [(0.9, 9), (0.95, 10)])
def test_most_harmonics(kpar, nr):
    """nr = 9 resonant harmonics, the most that tables hold (and the build's
    largest LDS), and one past it"""
    p = cases.kappa_case()
    t, _, lo, up = _tile(p, 0, kpar)
    om = _batch(p, 4000, 1.9 * t * kpar)
    assert math.ceil(np.max(om.real) + kpar * max(abs(lo), abs(up))) + 1 == nr
    _compare(p, om, 1 if nr <= 9 else 0, kpar)


def test_negative_kpar():
    """Im p = m Im om / kpar is positive for damped omegas: no tile covers it, and
    none is built"""
    p = cases.kappa_case()
    t, _, _, _ = _tile(p, 0)
    _compare(p, _batch(p, 1600, 1.9 * t * KPAR), 0, -KPAR)


@pytest.mark.parametrize("shape", [(8, 4, 4, 8, 2), (1, 4, 4, 4, 1)])
def test_species_without_tables_keep_their_lanes(shape):
    """The electrons' one resonant harmonic is not worth tables: their row sums take
    the shape's lanes, with the protons' tables (800 omegas) and without any (400),
    so their chi is the same to the last bit"""
    from alps_amd.engine import Engine
    p = cases.kappa_case()
    t, _, _, _ = _tile(p, 0)
    om = _batch(p, 800, 0.99 * t * KPAR)
    E = Engine(p)
    E.set_k(KPERP, KPAR)
    E.set_sweep_series(False)
    for n in (800, 400):
        E.set_shape(n, shape)
    assert E.landau_work(om)[0] == 1 and E.landau_work(om[:400])[0] == 0
    chi = [np.asarray(E.disp_batch(om[:n], want_tensors=True)[1])[:384, 1] for n in (800, 400)]
    E.close()
    assert np.array_equal(*chi)


@pytest.mark.parametrize("form", ["at", "below", "deep", "no_norm", "nan"])
def test_rule_edges(form):
    p = cases.kappa_two_fits()
    t, harm, lo, up = _tile(p, 0)
    n0 = max(512, math.ceil(64 * 64 * 2 / harm))
    depth = 1.9 * t * KPAR
    if form == "no_norm":
        p = dataclasses.replace(p, kperp_norm=False)
    om = _batch(p, n0 - (form == "below"), depth)
    if form == "deep":  # one omega past the last tile row: no tables for this species
        om[6] = 0.5 - 1j * 24.5 * t * KPAR
    if form == "nan":
        om[9:12] = complex(np.nan, 0.1), complex(0.2, np.nan), complex(np.nan, np.nan)
    # resonances at the ends of the accepted momenta
    om[7] = KPAR * lo + 0.5j * om[1].imag
    om[12] = KPAR * up * (1 - 1e-15) + 0.5j * om[1].imag
    _compare(p, om, 0 if form in ("below", "deep") else 1)
