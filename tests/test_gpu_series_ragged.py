"""GPU: every sample of partly filled waves.

A wave of the series takes the smallest step of its 64 rays, lanes without a
pixel included as harmless rays, so the last pixels of a ragged image have
other steps than in a whole one: their samples are held against direct
evaluation, not against another image's bits."""

import numpy as np
import pytest

from .kgeo_testlib import errors

pytestmark = pytest.mark.gpu
R_O = 1.0e4


@pytest.mark.parametrize("npix,ngeo", [(1, 3), (1, 250), (3, 40), (63, 17), (65, 18), (129, 40), (1000, 130), (4099, 9)])
def test_ragged_waves_match_direct_evaluation(npix, ngeo):
    """2e-11 normwise, and 100 times the direct evaluation's own move under a
    1e-14 change of tau where that is above 1e-12 (as test_series.py).  At the
    observer itself t and sigma are 0, which the series starts from exactly and
    the direct formulas miss by the rounding of r (up to 2e-10 of a ray next to
    the critical curve, where the rounded roots place the observer)."""
    import torch
    from kgeo_amd.raytrace import coords_at_tau_device, raytrace_ana_device
    a, th = 0.8, np.deg2rad(50.0)
    rng = np.random.default_rng(npix)
    A, B = rng.uniform(-7.0, 7.0, npix), rng.uniform(-7.0, 7.0, npix)
    g = raytrace_ana_device(a, R_O, th, A, B, ngeo)

    def direct(tau):
        sig, (t, r, thd, ph) = coords_at_tau_device(a, R_O, th, A, B, tau)
        return {k: v.cpu().numpy() for k, v in dict(t=t, r=r, th=thd, ph=ph, sig=sig).items()}

    ref, near = direct(g.tau), [direct(g.tau * f) for f in (1.0 + 1.0e-14, 1.0 - 1.0e-14)]
    torch.cuda.synchronize()
    for k in ("r", "th", "ph", "t", "sig"):
        x = getattr(g, k).cpu().numpy()
        assert np.array_equal(np.isnan(x), np.isnan(ref[k])), k
        e = np.nan_to_num(errors(x, ref[k], k))
        if k in ("t", "sig"):
            assert np.all(x[0] == 0.0), k
            e[0] = 0.0
        sens = np.max([np.nan_to_num(errors(n[k], ref[k], k)) for n in near], axis=0)
        assert np.all(e < np.where(sens > 1e-12, 100.0 * sens, 0.0) + 2e-11), (k, float(e.max()))
