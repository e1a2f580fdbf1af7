"""The linspace grid by Taylor series (kgeo_amd/csrc/kg_series_pass.hpp) on the
CPU build of the kernels' source, against direct evaluation of every sample.

The sizes are the edges of the pass: grids of 3 samples, below and above one
queued range and of one range per block and part, blocks of unequal length, one
part and the most; and the motions its formulas tell apart: both signs of the spin
and none, |a| below the reference's minimum (where case 3 loses a term),
near-equatorial, near-polar and vortical rays, rays next to the axis, and
rays of all three radial cases up to the horizon."""

import numpy as np
import pytest

from .kgeo_testlib import Host, errors, grid

CASES = [  # a, inclination, half window, pixels per side, samples, parts per block
    (0.94, 17.0, 8.0, 32, 500, 2),
    (0.94, 17.0, 8.0, 32, 500, 1),
    (0.94, 17.0, 1.0, 24, 250, 3),  # inside the shadow: radial cases 3 and 4
    (-0.6, 70.0, 7.0, 30, 37, 4),
    (0.99, 88.0, 8.0, 30, 130, 8),
    (0.5, 140.0, 6.0, 24, 17, 2),
    (0.3, 60.0, 5.0, 16, 3, 2),
    (0.3, 60.0, 5.0, 16, 8, 8),
    (0.3, 60.0, 5.0, 16, 9, 8),
    (0.0, 60.0, 8.0, 24, 120, 2),
    (5.0e-5, 45.0, 8.0, 24, 80, 3),
    (0.99, 5.0, 0.6, 24, 64, 2),  # vortical rays
    (-0.3, 3.0, 12.0, 40, 30, 1),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"a{c[0]}_th{c[1]}_w{c[2]}_G{c[4]}_p{c[5]}")
def test_series_matches_direct_evaluation(case):
    """Tolerances as for the walk (test_walk.py): 2e-11 normwise, and where the
    direct evaluation itself moves by more than 1e-12 under a 1e-14 relative
    change of tau, 100 times that move plus 2e-11.  The status words, the NaN
    pattern and the Mino times are the same, and splitting the blocks into
    parts changes no bit."""
    a, thd, w, n, G, parts = case
    A, B = grid(w, n)
    th = np.deg2rad(thd)
    host = Host()
    ser = host.raytrace_loops(a, 1.0e4, th, A, B, G, chunks=parts, passes=4)
    ref = host.raytrace_loops(a, 1.0e4, th, A, B, G, chunks=1, passes=1)
    assert np.array_equal(ser["tau"], ref["tau"])
    direct = host.raytrace_loops(a, 1.0e4, th, A, B, G, tau_in=ser["tau"])
    nudged = host.raytrace_loops(a, 1.0e4, th, A, B, G, tau_in=ser["tau"] * (1.0 + 1.0e-14))
    assert np.array_equal(ser["status"], direct["status"])
    whole = host.raytrace_loops(a, 1.0e4, th, A, B, G, chunks=1, passes=4)
    # hardly any range is left to direct evaluation (G/8 ranges per ray)
    assert ser["nfix"][0] < 0.02 * len(A) * (G / 8.0), ser["nfix"]
    for k in ("r", "th", "ph", "t", "sig"):
        assert np.array_equal(ser[k], whole[k], equal_nan=True), k
        assert np.array_equal(np.isnan(ser[k]), np.isnan(direct[k])), k
        e = np.nan_to_num(errors(ser[k], direct[k], k))
        sens = np.nan_to_num(errors(nudged[k], direct[k], k))
        assert np.all(e < np.where(sens > 1e-12, 100.0 * sens, 0.0) + 2e-11), (k, float(e.max()))
