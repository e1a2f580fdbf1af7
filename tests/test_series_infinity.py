"""Observers at infinity (r_o = inf, which the reference's raytrace_ana
accepts): r, theta and phi by the series as for any other; t and sigma, whose
terms are infinite, keep the reference's constant of each ray: infinite, NaN
or about 1e16.  CPU build of the kernels' source against direct evaluation."""

import numpy as np
import pytest

from .kgeo_testlib import Host, errors, grid


@pytest.mark.parametrize("G,parts", [(3, 1), (4, 1), (12, 2), (100, 3)])
@pytest.mark.parametrize("a,thd", [(0.7, 30.0), (-0.9, 75.0), (0.2, 120.0), (5.0e-5, 40.0), (0.0, 60.0)])
def test_series_from_infinity_matches_direct_evaluation(a, thd, G, parts):
    """r, theta and phi as in test_series.py (2e-11, and 100 times the direct
    evaluation's own move under a 1e-14 change of tau where that is above
    1e-12); status words and NaN and infinity patterns the same; finite t and
    sigma, a ray's constant but for O(1e4) changes, to 1e-11 of it away from
    the first sample (there the difference of the infinite terms' rounding);
    and hardly any range left to direct evaluation (all of 3 samples)."""
    A, B = grid(7.0, 40)
    A = A + 0.07
    host, th = Host(), np.deg2rad(thd)
    ser = host.raytrace_loops(a, np.inf, th, A, B, G, chunks=parts, passes=4)
    whole = host.raytrace_loops(a, np.inf, th, A, B, G, chunks=1, passes=5)
    direct = host.raytrace_loops(a, np.inf, th, A, B, G, tau_in=ser["tau"])
    nudged = host.raytrace_loops(a, np.inf, th, A, B, G, tau_in=ser["tau"] * (1.0 + 1.0e-14))
    assert np.array_equal(ser["status"], direct["status"])
    assert G == 3 or ser["nfix"][0] - len(A) < 0.02 * len(A) * (G / 8.0), ser["nfix"]
    for k in ("r", "th", "ph", "t", "sig"):
        assert np.array_equal(ser[k], whole[k], equal_nan=True), k
        assert np.array_equal(np.isnan(ser[k]), np.isnan(direct[k])), k
        assert np.array_equal(np.isinf(ser[k]), np.isinf(direct[k])), k
        if k in ("t", "sig"):
            ok = np.isfinite(direct[k])
            assert np.allclose(ser[k][ok], direct[k][ok], rtol=1e-11, atol=0.0), k
            continue
        e = np.nan_to_num(errors(ser[k], direct[k], k))
        sens = np.nan_to_num(errors(nudged[k], direct[k], k))
        assert np.all(e < np.where(sens > 1e-12, 100.0 * sens, 0.0) + 2e-11), (k, float(e.max()))


@pytest.mark.gpu
def test_gpu_rays_from_infinity():
    """The kernels, plain and batched: finite, infinite and NaN where direct
    evaluation at the same Mino times is, status words too; r and theta to 1e-10 of it."""
    import torch
    from kgeo_amd.batch import BatchSurvey
    from kgeo_amd.raytrace import coords_at_tau_device, raytrace_ana_device
    a, th, G = 0.7, np.deg2rad(30.0), 60
    A, B = grid(7.0, 48)
    A = A + 0.07
    g = raytrace_ana_device(a, np.inf, th, A, B, G)
    sig, (t, r, thd, ph) = coords_at_tau_device(a, np.inf, th, A, B, g.tau)
    sv = BatchSurvey([dict(a=a, th_o=th, alpha=A, beta=B, ngeo=G)], r_o=float("inf"), tuning=(64, 8))
    sv.run()
    sv.stream.synchronize()
    torch.cuda.synchronize()
    assert torch.equal(g.status, sv.status)
    for k, y in (("t", t), ("r", r), ("th", thd), ("ph", ph), ("sig", sig)):
        y = y.cpu().numpy()
        for x in (getattr(g, k), sv.arena[k].reshape(G, -1) if k != "sig" else g.sig):
            x = x.cpu().numpy()
            assert np.array_equal(np.isnan(x), np.isnan(y)) and np.array_equal(np.isinf(x), np.isinf(y)), k
            if k in ("r", "th"):
                assert np.nanmax(errors(x, y, k)[:-1]) < 1e-10, k
    sv.close()
