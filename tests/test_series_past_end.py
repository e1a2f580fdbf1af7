"""Rays followed past their end, backwards, and through the horizon (the
caller's maxtaufrac), on the CPU build of the kernels' source against direct
evaluation of every sample: grids that put a sample of every captured ray on
the horizon itself (maxtaufrac j / (ngeo - 1) = 1), where the closed forms of
the series are 0 times infinity, and ones that do not."""

import numpy as np
import pytest

from .kgeo_testlib import Host, errors, grid

R_O = 1.0e4
OBSERVERS = [(0.7, 40.0), (-0.9, 75.0), (0.2, 120.0)]
FRACS = [(1.5, 13), (1.5, 100), (4.0 / 3.0, 13), (1.25, 101), (1.0 + 1.0e-9, 40), (1.0, 40), (3.0, 13), (-0.5, 13),
         (-0.01, 40)]


@pytest.mark.parametrize("frac,ngeo", FRACS)
@pytest.mark.parametrize("a,thd", OBSERVERS)
def test_rays_past_their_end_match_direct_evaluation(a, thd, frac, ngeo, monkeypatch):
    """As test_series.py: 2e-11 normwise, and 100 times the direct evaluation's
    own move under a 1e-14 change of tau where that is above 1e-12; the same
    status words and the same NaN and infinity patterns."""
    scalars = Host.scalars
    monkeypatch.setattr(Host, "scalars", staticmethod(lambda *args: scalars(*args, frac)))
    A, B = grid(4.0, 48)
    A = A + 0.05
    host, th = Host(), np.deg2rad(thd)
    for parts in (1, 3):
        ser = host.raytrace_loops(a, R_O, th, A, B, ngeo, chunks=parts, passes=5)
        direct = host.raytrace_loops(a, R_O, th, A, B, ngeo, tau_in=ser["tau"])
        nudged = [host.raytrace_loops(a, R_O, th, A, B, ngeo, tau_in=ser["tau"] * f) for f in (1 + 1e-14, 1 - 1e-14)]
        assert np.array_equal(ser["status"], direct["status"])
        for k in ("r", "th", "ph", "t", "sig"):
            assert np.array_equal(np.isnan(ser[k]), np.isnan(direct[k])), k
            assert np.array_equal(np.isinf(ser[k]), np.isinf(direct[k])), k
            ok = np.isfinite(direct[k])
            x, y = (np.where(ok, v, 0.0) for v in (ser[k], direct[k]))
            with np.errstate(all="ignore"):
                e = np.where(ok, errors(x, y, k), 0.0)
                sens = np.max([np.nan_to_num(errors(np.where(ok, n[k], 0.0), y, k), nan=1.0) for n in nudged], axis=0)
            # t and sigma start at exactly 0 in the series, at the rounding of r_o in the direct formulas
            if k in ("t", "sig"):
                e[0] = np.where(np.abs(ser[k][0]) == 0.0, 0.0, e[0])
            bound = np.where(sens > 1e-12, 100.0 * sens, 0.0) + 2e-11
            assert np.all(e < bound), (k, float((e / bound).max()), np.argwhere(e / bound == (e / bound).max())[0])


@pytest.mark.gpu
@pytest.mark.parametrize("frac,ngeo", [(1.5, 13), (1.5, 100), (3.0, 13), (-0.5, 13)])
def test_gpu_rays_past_their_end(frac, ngeo):
    """The kernels on the same calls: finite where direct evaluation at the same
    Mino times is, r to 1e-10 of it and phi to 1e-8 of the ray (the direct
    formulas' own rounding next to the horizon, 2e-9 in the cases above)."""
    from kgeo_amd.raytrace import coords_at_tau_device, raytrace_ana_device
    a, th = 0.7, np.deg2rad(40.0)
    A, B = grid(4.0, 48)
    A = A + 0.05
    g = raytrace_ana_device(a, R_O, th, A, B, ngeo, maxtaufrac=frac)
    sig, (t, r, thd, ph) = coords_at_tau_device(a, R_O, th, A, B, g.tau)
    for k, x, y, tol in (("r", g.r, r, 1e-10), ("th", g.th, thd, 1e-10), ("ph", g.ph, ph, 1e-8)):
        x, y = x.cpu().numpy(), y.cpu().numpy()
        assert np.array_equal(np.isfinite(x), np.isfinite(y)), k
        ok = np.isfinite(y)
        with np.errstate(all="ignore"):
            e = np.where(ok, errors(np.where(ok, x, 0.0), np.where(ok, y, 0.0), k), 0.0)
        assert np.nanmax(e) < tol, (k, float(np.nanmax(e)))
