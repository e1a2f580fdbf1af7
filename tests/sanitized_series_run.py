"""Runs the series passes of the CPU build under AddressSanitizer and
UndefinedBehaviorSanitizer (kgeo_amd/libkgeo_hostcheck_san.so): the heads,
the blocks and their parts, early or not, and the fixups, over the grid lengths
where their indices change and the rays that queue ranges.  The build also
checks that no sample is queued twice and that the queue holds them all
(nfix).  Started by tests/test_sanitized_series.py in a child process whose
LD_PRELOAD holds the sanitizer runtime; any report aborts it."""

import ctypes
import os
import sys

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
sys.path.insert(0, ROOT)

from tests.kgeo_testlib import Host  # noqa: E402


def run():
    plain = Host()
    san = Host.__new__(Host)
    san.lib = ctypes.CDLL(os.path.join(ROOT, "kgeo_amd", "libkgeo_hostcheck_san.so"))
    scalars = Host.scalars
    rng = np.random.default_rng(12)
    # spin, inclination, window, r_o, maxtaufrac
    cases = [(0.94, 17.0, 8.0, 1e4, 1 - 1e-10), (-0.9, 80.0, 7.0, 1e4, 1 - 1e-10), (0.0, 60.0, 6.0, 1e4, 1 - 1e-10),
             (5e-5, 45.0, 6.0, np.inf, 1 - 1e-10), (0.99999, 30.0, 4.0, 1e4, 1 - 1e-10),
             (0.5, 140.0, 9.0, 100.0, 1.5), (0.7, 1e-9, 6.0, 1e4, 1 - 1e-10), (0.7, 40.0, 5.0, np.inf, 1.2)]
    checked = 0
    for a, th_deg, w, r_o, frac in cases:
        Host.scalars = staticmethod(lambda x, r, t: scalars(x, r, t, frac))
        th = th_deg * np.pi / 180
        npix = int(rng.integers(37, 90))
        al, be = rng.uniform(-w, w, npix), rng.uniform(-w, w, npix)
        al[:4], be[:4] = [0.0, 0.0, 1e-9, -w], [w, 0.3, 0.0, 1e-9]  # lambda = 0, next to the axis and the equator
        for ngeo in (3, 4, 5, 8, 9, 15, 16, 17, 18, 33, 100, 257):
            for parts in (1, 3, 8):
                for passes in (4, 5):
                    x, y = (h.raytrace_loops(a, r_o, th, al, be, ngeo, chunks=parts, passes=passes)
                            for h in (plain, san))
                    assert x["nfix"][0] >= 0 and y["nfix"][0] >= 0
                    for k in ("r", "th"):
                        # the builds contract differently; the last sample of captured rays is ill-conditioned
                        ok = np.isfinite(x[k][1:-1]) & np.isfinite(y[k][1:-1])
                        d = np.where(ok, np.abs(x[k][1:-1] - y[k][1:-1]) / np.maximum(np.abs(x[k][1:-1]), 1.0), 0.0)
                        assert d.max(initial=0.0) < 1e-5, (a, th_deg, ngeo, parts, passes, k, float(d.max()))
                    checked += 1
    print(f"sanitized series runs clean: {checked} pass configurations", flush=True)


if __name__ == "__main__":
    run()
