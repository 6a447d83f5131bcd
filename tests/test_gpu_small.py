"""Batches of at most 16 omegas, whose sums are assembled by the launch's last
workgroup: against the oracle and against the chain of separate kernels (which a
call for the tensors takes), on both sides of the staged assembly and in turns of
different sizes, so that a counter or a partial sum left by one launch would show
in the next.

Bar: 1e-11 of the determinant's terms (tests/test_gpu_disp.py).  Roots: secant_osc
stops at a step below D_prec, so D_prec of the root."""
import numpy as np
import pytest

import cases
from oracle import Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case", ["small_bimax", "three_species", "kappa_poly_mix"])
def test_sizes_in_turn(case):
    from alps_amd.engine import Engine
    p = getattr(cases, case)()
    E, O = Engine(p), Oracle(p)
    rng = np.random.default_rng(7)
    om = rng.uniform(0.05, 1.7, 17) + 1j * rng.uniform(-0.2, 0.1, 17)
    for kperp, kpar in ((0.3, 0.4), (0.7, 0.2)):
        E.set_k(kperp, kpar)
        O.set_k(kperp, kpar)
        for n in (1, 16, 2, 3, 15, 1, 17, 4, 16):
            det = E.disp_batch(om[:n])
            full = E.disp_batch(om[:n], want_tensors=True)
            sc = np.array([cases.det_scale(w) for w in np.asarray(full[3])])
            assert np.all(np.abs(det - full[0]) <= 1e-11 * sc), n
        for k in range(3):
            d, _, _, wave = O.disp(om[k], want_tensors=True)
            assert abs(E.disp_batch(om[k:k + 1])[0] - d) <= 1e-11 * cases.det_scale(wave)
    E.close()


def test_roots_in_turn():
    from alps_amd.engine import Engine
    p = cases.small_bimax()
    E = Engine(p)
    E.set_k(0.3, 0.4)
    root = E.secant_osc(0.4 - 0.01j)[0]
    for n in (1, 3, 16, 2, 17, 1):
        om, _, _ = E.secant_osc_batch(root * (1.0 + 1e-3 * np.exp(1j * np.arange(n))))
        assert np.all(np.abs(om - root) <= p.roots.D_prec), n
    E.close()


@pytest.mark.parametrize("case", ["kappa_case", "poly_case", "kappa_poly_mix"])
def test_roots_of_every_landau_form(case):
    """secant rounds of one launch (kappa fits alone) and of two (a species with the
    general Landau form) against the solves stepped on the host: the same steps to
    rounding, so well within the D_prec that ends them"""
    from alps_amd.engine import Engine
    p = getattr(cases, case)()
    E = Engine(p)
    E.set_k(0.3, 0.4)
    for n in (1, 3, 16, 2, 17, 1):
        g = 0.4 - 0.01j + 2e-3 * np.exp(1j * np.arange(n))
        om, _, it = E.secant_osc_batch(g)
        E.set_plain_roots(True)
        ref, _, it_ref = E.secant_osc_batch(g)
        E.set_plain_roots(False)
        assert np.array_equal(it, it_ref) and np.all(np.abs(om - ref) <= p.roots.D_prec), n
    E.close()
