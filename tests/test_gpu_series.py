"""GPU: the sample passes at the sizes where their launch shapes change."""

import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
R_O = 1.0e4


def _screen(n, a):
    rng = np.random.default_rng(n)
    return rng.uniform(-7.0, 7.0, n), rng.uniform(-7.0, 7.0, n)


@pytest.mark.parametrize("npix,ngeo", [(1, 3), (63, 17), (64, 18), (129, 40), (4096, 9), (20000, 41), (65000, 24)])
def test_samples_do_not_depend_on_the_number_of_pixels(npix, ngeo):
    """A ray's blocks are split into more parts the fewer pixels are sampled
    together: the first whole waves of a large image (one part) and the same
    pixels alone (up to eight) give the same bits, from grids below two queued
    ranges to several per part."""
    from kgeo_amd.raytrace import raytrace_ana_device
    a, th = 0.8, np.deg2rad(50.0)
    A, B = _screen(140000, a)
    whole = raytrace_ana_device(a, R_O, th, A, B, ngeo)
    g = raytrace_ana_device(a, R_O, th, A[:npix], B[:npix], ngeo)
    same = npix // 64 * 64 if npix >= 64 else 0  # a ragged wave has other neighbours
    for k in ("tau", "t", "r", "th", "ph", "sig"):
        x, y = getattr(g, k).cpu().numpy(), getattr(whole, k).cpu().numpy()[:, :npix]
        assert np.array_equal(np.isnan(x), np.isnan(y)), k
        assert np.array_equal(x[:, :same], y[:, :same], equal_nan=True), k
        # the first and the last sample are evaluated directly, whatever the wave
        for j in (0, -1):
            assert np.array_equal(x[j], y[j], equal_nan=True), (k, j)


@pytest.mark.parametrize("npix,ntau", [(1, 1), (64, 2), (65, 13), (500, 37)])
def test_direct_loops_do_not_depend_on_the_chunks(npix, ntau):
    """Caller-given Mino times: one lane per sample, per few samples and per
    pixel give the same bits."""
    import torch
    from kgeo_amd.raytrace import coords_at_tau_device
    a, th = 0.8, np.deg2rad(50.0)
    A, B = _screen(npix, a)
    tau = torch.from_numpy(np.random.default_rng(ntau).uniform(0.0, 0.1, (ntau, npix))).cuda()
    old = os.environ.get("KGEO_CHUNKS")
    got = []
    try:
        for c in (None, "1", "3"):
            os.environ.pop("KGEO_CHUNKS", None)
            if c:
                os.environ["KGEO_CHUNKS"] = c
            s, x = coords_at_tau_device(a, R_O, th, A, B, tau)
            got.append([s] + list(x))
    finally:
        os.environ.pop("KGEO_CHUNKS", None)
        if old is not None:
            os.environ["KGEO_CHUNKS"] = old
    for other in got[1:]:
        for x, y in zip(got[0], other):
            assert np.array_equal(x.cpu().numpy(), y.cpu().numpy(), equal_nan=True)
