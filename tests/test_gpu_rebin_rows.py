"""Rebinning where its kernels change course: rows that just fit LDS and the
first that do not, one launch and two, the smallest scans, more detectors than a block has lanes,
and view angles far from evenly spaced (the guessed intervals miss), and the output
over the input.  And the helical interpolation over fan angles and view counts
that move its rounded views.  Bit for bit against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("even", [True, False])
@pytest.mark.parametrize("geom", [1, 2])
@pytest.mark.parametrize("nDet,nView", [(2, 2), (3, 3), (64, 65), (513, 40), (1025, 6), (1025, 256), (1537, 511),
                                        (2049, 512), (5120, 6), (5120, 512), (5121, 6)])
def test_rebin_rows(gpu_ctx, oracle_lib, geom, nDet, nView, even):
    import torch
    import ctsim_amd
    print(f"case rebin rows geom={geom} {nDet}x{nView} even={even}", flush=True)
    rng = np.random.default_rng(nDet + nView)
    data = rng.standard_normal((nView, nDet)).astype(np.float32)
    F, sdl, vd = 2.0, 4.0, 2.0
    fan = 2 * np.arcsin(vd / 2 / F)
    detInc = fan / nDet if geom == 1 else 2 * sdl * np.tan(fan / 2) / nDet
    angles = np.arange(nView) * (2 * np.pi / nView) if even else np.sort(rng.uniform(0, 1, nView) ** 6 * 2 * np.pi)
    info6 = [-(nDet - 1) / 2 * detInc, detInc, F, sdl, vd, 0.0]
    ref, rang, _ = oracle_lib.interpolate_to_parallel(geom, data, *info6, angles)
    r = ctsim_amd.Rebin(gpu_ctx, geom, nDet, nView, *info6, angles)
    out = r.run(torch.from_numpy(data).cuda()).cpu().numpy()
    assert np.array_equal(out.view(np.uint32), ref.view(np.uint32))
    assert np.array_equal(r.angles, rang)


@pytest.mark.parametrize("shift", [0, 1, -3])
@pytest.mark.parametrize("nDet,nView", [(64, 65), (513, 400), (2049, 512), (5121, 6)])
def test_rebin_in_place(gpu_ctx, nDet, nView, shift):
    """Output over the input, or `shift` rows beside it, and several runs on:
    what two buffers give."""
    import ctypes as C
    import torch
    import ctsim_amd
    from ctsim_amd import api
    print(f"case rebin in place {nDet}x{nView} shift {shift}", flush=True)
    F, sdl, vd = 2.0, 4.0, 2.0
    detInc = 2 * np.arcsin(vd / 2 / F) / nDet
    angles = np.arange(nView) * (2 * np.pi / nView)
    r = ctsim_amd.Rebin(gpu_ctx, 1, nDet, nView, -(nDet - 1) / 2 * detInc, detInc, F, sdl, vd, 0.0, angles)
    buf = torch.zeros((nView + 6, nDet), dtype=torch.float32, device="cuda")
    for seed in range(3):
        sino = torch.from_numpy(np.random.default_rng(seed).standard_normal((nView, nDet)).astype(np.float32)).cuda()
        want = r.run(sino)
        src, dst = buf[3:3 + nView], buf[3 + shift:3 + shift + nView]
        src.copy_(sino)
        rc = api.lib.ctsim_rebin_run(gpu_ctx.handle, r.handle, C.c_void_p(src.data_ptr()), C.c_void_p(dst.data_ptr()))
        api.check(rc, "ctsim_rebin_run")
        torch.cuda.synchronize()
        assert torch.equal(dst.view(torch.int32), want.view(torch.int32))


@pytest.mark.parametrize("geom", [1, 2])
@pytest.mark.parametrize("nDet,nView,fan", [(7, 90, 0.3), (64, 181, 1.9), (129, 360, 0.01), (300, 777, 1.0)])
def test_helical_views(gpu_ctx, oracle_lib, geom, nDet, nView, fan):
    import torch
    import ctsim_amd
    print(f"case helical views geom={geom} {nDet}x{nView} fan={fan}", flush=True)
    rng = np.random.default_rng(nDet)
    data = rng.standard_normal((nView, nDet)).astype(np.float32)
    rotInc, sdl = (2 * (np.pi + fan) + 0.2) / nView, 4.0
    detInc = fan / nDet if geom == 1 else 2 * sdl * np.tan(fan / 2) / nDet
    for feather in (False, True):
        ref, _ = oracle_lib.helical180li(geom, data, rotInc, detInc, fan, sdl, -1, feather)
        out, _ = ctsim_amd.helical180li(gpu_ctx, geom, torch.from_numpy(data).cuda(), rotInc, detInc, fan, sdl, -1)
        if feather:
            out = ctsim_amd.halfscan_feather(gpu_ctx, geom, out, rotInc, detInc, fan, sdl)
        assert np.array_equal(out.cpu().numpy().view(np.uint32), ref.view(np.uint32))
