"""Block 0 of the series as the plain kernels run it, beside the radial half of
the plan (which it must not read), on the CPU build of their source: the same
samples, status and queued ranges as the block run after it, which is what
the batched survey does."""

import numpy as np
import pytest

from .kgeo_testlib import Host, grid
from .test_series import CASES

R_O = 1.0e4
KEYS = ("tau", "t", "r", "th", "ph", "sig", "status")

# Pixels on the critical curve, found by bisection (a, inclination, alpha, beta):
# within a few ulp of alpha the two outer roots of some round to one, radial
# modulus 1, which neither the heads nor the series serve.
CRITICAL = [(0.5, 60.0, 5.791643817227586, 1.472403584600264), (0.5, 60.0, 5.537634861155227, -2.1548623280500205),
            (0.5, 60.0, 5.985843999000293, 0.43272401738614263), (0.5, 60.0, 4.981801949463874, -3.0990906756755425),
            (0.5, 60.0, 4.816272436314191, 3.310701341385303), (0.5, 60.0, 5.592913470128523, -2.0287522475921955)]


def _same(x, y):
    for k in KEYS:
        assert np.array_equal(x[k], y[k], equal_nan=x[k].dtype.kind == "f"), k
    assert np.array_equal(x["nfix"], y["nfix"])


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"a{c[0]}_th{c[1]}_w{c[2]}_G{c[4]}_p{c[5]}")
def test_early_block_gives_the_same_bits(case):
    a, thd, w, n, G, parts = case
    A, B = grid(w, n)
    host, th = Host(), np.deg2rad(thd)
    _same(host.raytrace_loops(a, R_O, th, A, B, G, chunks=parts, passes=5),
          host.raytrace_loops(a, R_O, th, A, B, G, chunks=parts, passes=4))


@pytest.mark.parametrize("G", [4, 17, 100])
def test_rays_of_modulus_one_are_direct_in_every_block(G):
    """Beside an ordinary pixel: the same samples whether block 0 runs early or
    not, and where the whole ray is left to direct evaluation (its last sample
    too, which a served ray's head writes) the direct samples."""
    host = Host()
    last = G - 1
    windows = sum(-(-e // 8) - s // 8 for s, e in ((0, (last + 1) // 2), ((last + 1) // 2, G)))
    whole = 0
    for a, thd, al, be in CRITICAL:
        for d in range(-4, 5):
            A, B, th = np.array([al + d * np.spacing(al), 3.0]), np.array([be, 1.0]), np.deg2rad(thd)
            early = host.raytrace_loops(a, R_O, th, A, B, G, passes=5)
            _same(early, host.raytrace_loops(a, R_O, th, A, B, G, passes=4))
            if early["nfix"][0] < windows or (G - 1) % 8:
                continue
            whole += 1
            direct = host.raytrace_loops(a, R_O, th, A, B, G, tau_in=early["tau"])
            for k in KEYS:
                assert np.array_equal(early[k][..., 0], direct[k][..., 0], equal_nan=early[k].dtype.kind == "f"), k
    assert whole >= (10 if G == 17 else 0)


@pytest.mark.gpu
def test_plain_and_batched_agree_on_rays_of_modulus_one():
    """The plain call (block 0 early) and the batched survey on the same rays,
    critical ones among ordinary ones: status words, NaN patterns, and both ends
    of each ray, which are direct or closed-form in either."""
    import torch
    from kgeo_amd.batch import BatchSurvey
    from kgeo_amd.raytrace import raytrace_ana_device
    a, thd = CRITICAL[0][:2]
    th = float(np.deg2rad(thd))
    al = np.array([x + d * np.spacing(x) for _, _, x, _ in CRITICAL for d in range(-4, 5)] + list(np.linspace(1.0, 9.0, 20)))
    be = np.array([b for _, _, _, b in CRITICAL for _ in range(9)] + list(np.linspace(-3.0, 3.0, 20)))
    for G in (4, 17, 40):
        plain = raytrace_ana_device(a, R_O, th, al, be, G)
        sv = BatchSurvey([dict(a=a, th_o=th, alpha=al, beta=be, ngeo=G)], r_o=R_O, tuning=(64, 8))
        sv.run()
        sv.stream.synchronize()
        torch.cuda.synchronize()
        assert torch.equal(plain.status, sv.status[:len(al)])
        for k in ("t", "r", "th", "ph"):
            x = getattr(plain, k).cpu().numpy()
            y = sv.arena[k][:G * len(al)].cpu().numpy().reshape(G, len(al))
            assert np.array_equal(np.isnan(x), np.isnan(y)), (G, k)
            for j in (0, G - 1):
                assert np.allclose(x[j], y[j], rtol=1e-12, atol=1e-12, equal_nan=True), (G, k, j)
        sv.close()
