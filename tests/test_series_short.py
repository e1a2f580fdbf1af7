"""Short grids of the series next to the critical curve (CPU build of the
kernels' source, against the oracle).

There a difference in the last bit grows along the ray, so no sample may be
more than half a ray from a direct evaluation, however few samples the grid
has: from three, over the sizes around one and two queued ranges (8 samples)
to the ones whose middle is furthest from a multiple of 8."""

import numpy as np
import pytest

from oracle import kgeo_oracle as O

from .kgeo_testlib import Host, conditioning_mask, errors, grid

R_O = 1.0e4
SCREENS = [(-0.712, 80.8, 7.57), (0.9, 60.0, 8.0), (0.94, 17.0, 8.0), (0.5, 30.0, 6.0)]


def _critical_pixels(host, a, th, w, n=400, keep=96):
    """The pixels of an n x n screen whose rays are longest in Mino time: the
    ones nearest the critical curve."""
    A, B = grid(w, n)
    stop = host.raytrace_loops(a, R_O, th, A, B, 2, passes=1)["tau"][-1]
    idx = np.sort(np.argsort(-np.nan_to_num(stop))[:keep])
    return A[idx], B[idx]


@pytest.mark.parametrize("ngeo", [3, 4, 5, 7, 8, 9, 10, 12, 16, 17, 32, 48])
@pytest.mark.parametrize("screen", SCREENS, ids=lambda s: f"a{s[0]}_th{s[1]}")
def test_short_grids_next_to_the_critical_curve(screen, ngeo):
    """Well-conditioned samples within 1e-10 of the oracle (conditioning_mask,
    the suite's parity bound), the last sample of captured rays left out by it;
    and splitting the blocks into parts changes no bit."""
    a, thd, w = screen
    th = np.deg2rad(thd)
    host = Host()
    A, B = _critical_pixels(host, a, th, w)
    got = host.raytrace_loops(a, R_O, th, A, B, ngeo, chunks=1, passes=4)
    parts = host.raytrace_loops(a, R_O, th, A, B, ngeo, chunks=8, passes=4)
    with np.errstate(all="ignore"):
        ref = O.raytrace_ana(a, R_O, th, A, B, ngeo)
        ill = conditioning_mask(a, R_O, th, A, B, ref["tau"], ref)
    assert np.count_nonzero(~ill) > 0.3 * ill.size
    for k in ("r", "th", "ph", "t", "sig"):
        assert np.array_equal(got[k], parts[k], equal_nan=True), k
        e = np.where(ill, 0.0, np.nan_to_num(errors(got[k], ref[k], k)))
        assert e.max() < 1e-10, (k, float(e.max()), np.argwhere(e == e.max())[0].tolist())
