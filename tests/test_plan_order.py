"""Every raytrace entry leaves its work ordered on the caller's stream.

The plan's radial constants run on a library-owned stream; a call that returns
without a sample pass behind them would leave them reading alpha and beta and
writing the workspace after the caller's stream is done.  Under stream capture
such a call cannot be captured (the capture would end unjoined)."""

import ctypes

import numpy as np
import pytest

from kgeo_amd import _lib


def test_missing_outputs_are_refused_before_the_plan():
    """t and ph are checked before anything is enqueued (without a GPU the
    plan's first launch would fail with KGEO_E_HIP instead)."""
    lib = _lib.load()
    buf = (ctypes.c_char * 8192)()
    fake = ctypes.c_void_p((ctypes.addressof(buf) + 255) // 256 * 256)
    p = _lib.make_params(0.5, 1e4, 0.5, 10, 10, 1.0)
    for t, ph in ((None, fake), (fake, None)):
        rcs = [
            lib.kgeo_raytrace_ana(ctypes.byref(p), fake, fake, None, t, None, None, ph, None, None, None, None, None,
                                  None, fake, 1 << 40, None),
            lib.kgeo_coords_at_tau(ctypes.byref(p), fake, fake, fake, 10, t, None, None, ph, None, None, fake,
                                   1 << 40, None),
            lib.kgeo_sample(ctypes.byref(p), None, 10, None, t, None, None, ph, None, None, fake, 1 << 40, None),
        ]
        assert rcs == [-1, -1, -1], rcs
        assert b"t and ph" in lib.kgeo_last_error()


@pytest.mark.gpu
@pytest.mark.parametrize("npix", [1, 700])
def test_a_plan_alone_can_be_captured(npix):
    """kgeo_plan and kgeo_coords_at_tau without Mino times, captured and
    replayed: the plan is the eager call's, whose samples then have the bits of
    kgeo_raytrace_ana."""
    import torch
    from kgeo_amd.raytrace import _ptr, _stream_handle, raytrace_ana_device
    lib = _lib.load()
    a, r_o, th, ngeo = 0.8, 1.0e4, 0.9, 20
    rng = np.random.default_rng(npix)
    al, be = (torch.from_numpy(rng.uniform(-7.0, 7.0, npix)).cuda() for _ in range(2))
    ref = raytrace_ana_device(a, r_o, th, al, be, ngeo)
    p = _lib.make_params(a, r_o, th, npix, ngeo, 1.0 - 1.0e-10)
    wsb = _lib.workspace_bytes(npix, ngeo)
    used = _lib.workspace_bytes(npix)
    ws = torch.zeros(wsb, device="cuda", dtype=torch.uint8)
    status = torch.zeros(npix, device="cuda", dtype=torch.int32)
    tau_tot = torch.zeros(npix, device="cuda", dtype=torch.float64)

    def plan():
        _lib.check(lib.kgeo_plan(p, _ptr(al), _ptr(be), None, None, None, _ptr(tau_tot), _ptr(status), _ptr(ws), wsb,
                                 _stream_handle()), "kgeo_plan")

    def coords():
        _lib.check(lib.kgeo_coords_at_tau(p, _ptr(al), _ptr(be), None, 0, None, None, None, None, None, _ptr(status),
                                          _ptr(ws), wsb, _stream_handle()), "kgeo_coords_at_tau")

    for call in (plan, coords):
        call()
        torch.cuda.synchronize()
        eager = ws[:used].cpu().numpy().copy()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            call()
        for _ in range(3):
            ws.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert np.array_equal(ws[:used].cpu().numpy(), eager)
    out = {k: torch.empty((ngeo, npix), device="cuda", dtype=torch.float64) for k in ("t", "r", "th", "ph")}
    _lib.check(lib.kgeo_sample(p, None, ngeo, None, _ptr(out["t"]), _ptr(out["r"]), _ptr(out["th"]), _ptr(out["ph"]),
                               None, _ptr(status), _ptr(ws), wsb, _stream_handle()), "kgeo_sample")
    for k, v in out.items():
        assert torch.equal(torch.nan_to_num(v, 7.0), torch.nan_to_num(getattr(ref, k), 7.0)), k
    assert torch.equal(tau_tot, ref.tau_tot)
