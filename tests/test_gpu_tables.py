"""The per-k tables where their launches can go wrong: pperp rows around the
groups they are loaded in (4, 16 and 64), harmonics around the 6 a workgroup of
J_n makes and the 16-row tiles, species with different harmonics, and the
split-form tables, which the first large batch of a k builds.

Bar: 1e-11 of the species' largest |chi| (tests/test_gpu_disp.py)."""
import numpy as np
import pytest

import cases
from oracle import Oracle

pytestmark = pytest.mark.gpu

TOL = 1e-11
OMS = [0.5113 + 0.0511j, 0.3127 - 0.0021j, 0.1217 + 0.3j, 1.5131 - 0.3j]


def _close(chi, low, ref):
    for k, (c, l) in enumerate(ref):
        for g, o in ((chi[k], c), (low[k], l)):
            for s in range(o.shape[0]):
                assert np.max(np.abs(g[s] - o[s])) <= TOL * np.max(np.abs(o[s])), (k, s)


@pytest.mark.parametrize("nperp,npar,kperp", [(4, 20, 0.3), (5, 31, 0.9), (16, 33, 0.05),
                                              (17, 34, 0.5), (18, 65, 1.7), (63, 64, 0.2),
                                              (64, 30, 0.7), (65, 37, 1.1), (130, 41, 0.01)])
def test_rows_and_harmonics(nperp, npar, kperp):
    from alps_amd.engine import Engine
    p = cases.three_species(nperp, npar)
    E, O = Engine(p), Oracle(p)
    # two k in turn: the second one's tables replace the first's, the lazily
    # built ones too
    for kp, kz in ((kperp, 0.3), (1.6 * kperp, 0.21)):
        assert E.set_k(kp, kz) == O.set_k(kp, kz)
        ref = [O.disp(om, want_tensors=True)[1:3] for om in OMS]
        _, chi, low, _ = E.disp_batch(np.array(OMS), want_tensors=True)
        _close(chi, low, ref)
        det = E.disp_batch(np.array(OMS))
        # the one-lane sweep of large batches
        _, chi, low, _ = E.disp_batch(np.resize(np.array(OMS), 2050), want_tensors=True)
        _close(chi, low, ref)
        big = E.disp_batch(np.resize(np.array(OMS), 2050))
        np.testing.assert_allclose(big[:4], det, rtol=1e-9)
        np.testing.assert_allclose(big[-2:], big[:2], rtol=1e-9)
    E.close()
