"""Parameter records of many lensed curves (kgeo_amd/lensing.py)."""

import numpy as np
import pytest


@pytest.mark.parametrize("n", [1, 2, 5, 17, 2000])
def test_curve_parameters_match_the_scalar_ones(n, monkeypatch):
    """The records, built over arrays, hold the bits of make_params for each curve."""
    import torch
    from kgeo_amd import _lib, lensing
    monkeypatch.setattr(lensing, "_device", lambda: torch.device("cpu"))
    rng = np.random.default_rng(n)
    spins, incs = rng.uniform(-0.99, 0.99, n), rng.uniform(0.01, 3.13, n)
    arr = (_lib.RayParams * n)()
    for k in range(n):
        arr[k] = _lib.make_params(float(spins[k]), lensing.R0, float(incs[k]), 1, 1, 1.0)
    assert bytes(arr) == lensing._curve_params(spins, incs).numpy().tobytes()
