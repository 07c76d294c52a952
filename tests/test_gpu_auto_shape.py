"""The launch shape that an untuned mixed slice takes (rotational, mirror or
plain kernel by the views' symmetry, rows per lane and view groups by size),
against the plain kernel with one view group on the same inputs.  Both form
FP32 positions relative to a window of up to 128 cells, each within an ulp or
two (2^-17 cells) of the exact one, and add compensated FP32 sums; rows of
white noise change by 1.4 of their size per cell, so one contribution of the
two differs by at most 4 x 2^-17 x 1.4 = 4.3e-5 of the rows' size, and the
images, over whose views the differences have either sign, by less than half
of that in norm: 2e-5.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TWO_PI = 2 * np.pi


def _angles(kind, nView, parallel):
    full = np.pi if parallel else TWO_PI
    a = np.arange(nView) * (full / nView)
    if kind == "back":
        return a[::-1].copy()
    if kind == "offset":
        return a + 0.3
    if kind == "shuffled":
        return np.random.default_rng(1).permutation(a)
    if kind == "half":
        return a * 0.6
    return a


def _plans(ctx, geom, nDet, nView, nx, ny, interp, roi=None):
    import ctsim_amd
    F = 2 * np.sqrt(2.0)
    a = np.arcsin(0.5)
    inc = {"parallel": 2 * np.sqrt(2.0), "equiangular": 2 * a, "equilinear": 4 * F * np.tan(a)}[geom] / nDet
    ps = ctsim_amd.ProcessSignal(ctx, "abs_hanning", "fft", 1 / inc, inc, nDet, geometry=geom, focalLength=F,
                                 sourceDetectorLength=2 * F)
    bp = ctsim_amd.Backprojector(ctx, geom, nDet, inc, nView, 2 * np.sqrt(2.0), F, 2 * F, "idiff", interp, nx, ny, roi)
    return ps, bp


# S = 4, S = 2 and no rotated copies; two, four and no mirrors; odd, rectangular and tiny images; one view
SHAPES = [("fan", 183, 90, 128, 128, "whole"), ("fan", 64, 1, 16, 16, "whole"), ("fan", 200, 181, 129, 129, "whole"),
          ("fan", 300, 360, 256, 256, "back"), ("fan", 300, 362, 200, 200, "offset"), ("fan", 129, 77, 90, 41, "whole"),
          ("fan", 300, 200, 150, 150, "half"), ("fan", 257, 160, 256, 256, "shuffled"), ("fan", 700, 240, 641, 640, "whole"),
          ("fan", 90, 500, 300, 300, "half"),
          # tall and wide images, two and four mirrors, 16 and 32 groups; windows of most of the detector
          ("fan", 210, 402, 40, 300, "whole"), ("fan", 210, 201, 300, 40, "whole"), ("fan", 150, 802, 300, 47, "whole"),
          ("fan", 180, 770, 47, 210, "whole"), ("fan", 120, 403, 230, 230, "whole"), ("fan", 400, 302, 16, 700, "whole")]


@pytest.mark.parametrize("interp", ["linear", "cubic"])
@pytest.mark.parametrize("geom", ["parallel", "equiangular", "equilinear"])
@pytest.mark.parametrize("_,nDet,nView,nx,ny,kind", SHAPES)
def test_auto_shape_matches_plain_kernel(gpu_ctx, _, geom, nDet, nView, nx, ny, kind, interp):
    import torch
    import ctsim_amd
    print(f"case auto shape {geom} {nDet}x{nView} {nx}x{ny} {kind} {interp}", flush=True)
    angles = _angles(kind, nView, geom == "parallel")
    rows = np.random.default_rng(nDet).standard_normal((nView, nDet)).astype(np.float32)
    sino = torch.from_numpy(rows).cuda()
    out = []
    for plain in (False, True):
        ps, bp = _plans(gpu_ctx, geom, nDet, nView, nx, ny, interp)
        if plain:
            bp.set_shape(16, 1, 1, 4, 0)
        img = torch.full((nx, ny), 7.0, dtype=torch.float32, device="cuda")
        bp.fbp(ps, sino, angles, img, ctsim_amd.PREC_MIXED)
        torch.cuda.synchronize()
        out.append(img.cpu().numpy().astype(np.float64))
    assert np.linalg.norm(out[0] - out[1]) <= 2e-5 * np.linalg.norm(out[1])


def test_region_of_interest(gpu_ctx):
    """A region away from the centre has no symmetry to use."""
    import torch
    import ctsim_amd
    angles = _angles("whole", 96, False)
    sino = torch.from_numpy(np.random.default_rng(0).standard_normal((96, 150)).astype(np.float32)).cuda()
    out = []
    for plain in (False, True):
        ps, bp = _plans(gpu_ctx, "equiangular", 150, 96, 100, 80, "linear", (-0.2, -0.9, 0.9, 0.3))
        if plain:
            bp.set_shape(16, 1, 1, 4, 0)
        img = torch.zeros((100, 80), dtype=torch.float32, device="cuda")
        bp.fbp(ps, sino, angles, img, ctsim_amd.PREC_MIXED)
        torch.cuda.synchronize()
        out.append(img.cpu().numpy().astype(np.float64))
    assert np.linalg.norm(out[0] - out[1]) <= 2e-5 * np.linalg.norm(out[1])


def test_static_scratch_takes_what_it_took(gpu_ctx):
    """A slice whose view groups' partial images exceed the static scratch
    (8 x 9 MB) runs there, and as ctsim_fbp_slice, with fewer groups."""
    import ctypes as C
    import torch
    import ctsim_amd
    from ctsim_amd import api
    nx, nDet, nView = 1500, 300, 255
    angles = _angles("whole", nView, False)
    sino = torch.from_numpy(np.random.default_rng(0).standard_normal((nView, nDet)).astype(np.float32)).cuda()
    ps, bp = _plans(gpu_ctx, "equilinear", nDet, nView, nx, nx, "linear")
    a = torch.zeros((nx, nx), dtype=torch.float32, device="cuda")
    b = torch.zeros_like(a)
    bp.fbp(ps, sino, angles, a, ctsim_amd.PREC_MIXED)
    rc = api.lib.ctsim_fbp_slice_static(gpu_ctx.handle, ps.handle, bp.handle, C.c_void_p(sino.data_ptr()),
                                        angles.ctypes.data_as(C.c_void_p), nView, C.c_void_p(b.data_ptr()))
    api.check(rc, "ctsim_fbp_slice_static")
    torch.cuda.synchronize()
    assert torch.equal(a.view(torch.int32), b.view(torch.int32))
