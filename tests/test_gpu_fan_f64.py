"""The FP64 fan-beam backprojection with linear and cubic interpolation
(backproject_f64.hip) where its dispatch and tiles end: image sizes around the
16-pixel tile, view counts around the 4 and 8 views taken at a time and the
128 whose constants are found together, every arc-tangent degree, detectors so
fine that the general kernel serves, rows of noise (whose contributions the
short formula leaves to the reference's own operations most often), zeros,
infinities and no numbers.  Every comparison is bit for bit."""
import numpy as np
import pytest

from conftest import record_parity
from ctsim_amd import workloads as W

pytestmark = pytest.mark.gpu


def _scan(O, geom, nDet, nView, scanRatio=1.0):
    return (O.Phantom(None, W.mixed_elements(31)),
            O.ScanSpec(geom, nDet, nView, 0, 1, 2 * np.pi, 2.0, 2.0, 1.0, scanRatio))


def _plan(ctx, geom, nDet, nView, nx, ny, interp, info):
    import ctsim_amd
    return ctsim_amd.Backprojector(ctx, geom, nDet, info["detInc"], nView, info["viewDiameter"],
                                   info["focalLength"], info["sourceDetectorLength"], "idiff", interp, nx, ny)


def _info(geom, nDet, nView, scanRatio=1.0):
    import ctsim_amd
    return ctsim_amd.Scanner(ctsim_amd.Phantom(None, W.mixed_elements(31)), geom, nDet, nView, 0, 1,
                             2 * np.pi, 2.0, 2.0, 1.0, scanRatio).info


# image, detectors, views, scan ratio (0.5: the detector ends inside the image): degree 14 (24, 40 and 64 pixels across), 8 (130, 200), 5 (320); the last row's
# windows are too long to stage, so the general kernel runs
SHAPES = [(16, 16, 65, 1, 1.0), (17, 33, 66, 7, 1.0), (24, 1, 65, 8, 1.0), (40, 64, 97, 9, 1.0),
          (130, 95, 200, 129, 1.0), (200, 33, 367, 12, 1.0), (320, 31, 500, 131, 1.0), (64, 50, 97, 33, 0.5),
          (33, 17, 1200, 5, 1.0), (20, 20, 3000, 4, 1.0)]


@pytest.mark.parametrize("interp", ["linear", "cubic"])
@pytest.mark.parametrize("geom", ["equiangular", "equilinear"])
@pytest.mark.parametrize("nx,ny,nDet,nView,scanRatio", SHAPES)
def test_noise_rows_match_oracle(gpu_ctx, oracle_lib, geom, interp, nx, ny, nDet, nView, scanRatio):
    import torch
    import ctsim_amd
    print(f"case fan f64 {geom} {interp} {nx}x{ny} {nDet}x{nView}", flush=True)
    phm, scan = _scan(oracle_lib, geom, nDet, nView, scanRatio)
    rows = np.random.default_rng(nx + nView).standard_normal((nView, nDet))
    angles = np.arange(nView) * (2 * np.pi / nView)
    want = oracle_lib.backproject("oracle", phm, scan, "idiff", interp, nx, ny, rows, angles)
    info = _info(geom, nDet, nView, scanRatio)
    b = _plan(gpu_ctx, geom, nDet, nView, nx, ny, interp, info)
    img = torch.zeros((nx, ny), dtype=torch.float32, device="cuda")
    b.backproject(torch.from_numpy(rows).cuda(), angles, img, ctsim_amd.PREC_F64)
    b.postprocess(img)
    torch.cuda.synchronize()
    assert record_parity(f"oracle fan f64 {geom} {interp} {nx}x{ny} {nDet}x{nView}", img.cpu().numpy(), want) == 0


@pytest.mark.parametrize("interp", ["linear", "cubic"])
@pytest.mark.parametrize("geom", ["equiangular", "equilinear"])
@pytest.mark.parametrize("kind", ["zeros", "inf", "nan", "tiny"])
def test_special_rows_match_general_kernel(gpu_ctx, geom, interp, kind):
    """Turning every view by five whole turns selects the general kernel and
    changes the positions by no more than their rounding, which these rows do
    not show: zeros onto pixels of either sign, one cell in each row that is
    infinite or no number, and contributions below the least float32."""
    import torch
    import ctsim_amd
    nx, ny, nDet, nView = 70, 45, 67, 11
    print(f"case fan f64 special {geom} {interp} {kind}", flush=True)
    rows = np.zeros((nView, nDet))
    if kind in ("inf", "nan"):
        rows[np.arange(nView), 20 + 2 * np.arange(nView)] = np.inf if kind == "inf" else np.nan
    elif kind == "tiny":
        rows[:] = 1e-60
    start = np.zeros((nx, ny), np.float32)
    start[::2] = -0.0
    angles = np.arange(nView) * (2 * np.pi / nView) + 0.01
    info = _info(geom, nDet, nView)
    out = []
    for turn in (0.0, 10 * np.pi):
        b = _plan(gpu_ctx, geom, nDet, nView, nx, ny, interp, info)
        img = torch.from_numpy(start.copy()).cuda()
        b.backproject(torch.from_numpy(rows).cuda(), angles + turn, img, ctsim_amd.PREC_F64)
        torch.cuda.synchronize()
        out.append(img.cpu().numpy())
    nan = np.isnan(out[0])
    assert np.array_equal(nan, np.isnan(out[1]))
    assert np.array_equal(out[0][~nan].view(np.uint32), out[1][~nan].view(np.uint32))


def test_views_in_parts_add_up(gpu_ctx):
    """Views added in two calls, the second onto the first one's image, give
    the image of one call."""
    import torch
    import ctsim_amd
    nDet, nView, nx = 129, 150, 90
    info = _info("equiangular", nDet, nView)
    b = _plan(gpu_ctx, "equiangular", nDet, nView, nx, nx, "cubic", info)
    rows = torch.from_numpy(np.random.default_rng(5).standard_normal((nView, nDet))).cuda()
    angles = np.arange(nView) * (2 * np.pi / nView)
    whole = torch.zeros((nx, nx), dtype=torch.float32, device="cuda")
    parts = torch.zeros_like(whole)
    b.backproject(rows, angles, whole, ctsim_amd.PREC_F64)
    b.backproject(rows[:61].contiguous(), angles[:61], parts, ctsim_amd.PREC_F64)
    b.backproject(rows[61:].contiguous(), angles[61:], parts, ctsim_amd.PREC_F64)
    torch.cuda.synchronize()
    assert torch.equal(whole.view(torch.int32), parts.view(torch.int32))


@pytest.mark.parametrize("interp", ["linear", "cubic"])
@pytest.mark.parametrize("geom", ["equiangular", "equilinear"])
@pytest.mark.parametrize("nx", [45, 64, 129])
def test_no_number_beside_a_cell_boundary(gpu_ctx, oracle_lib, geom, interp, nx):
    """Views at multiples of 45 degrees put a square image's middle row,
    column or diagonal on the centre cell to within rounding, so that the
    reference reads either of two intervals there: a cell that is no number
    in the one beside the interval of the short formula's position reaches the
    pixel or not as the reference's own operations decide."""
    import torch
    import ctsim_amd
    nDet = 67
    print(f"case fan f64 no number beside a boundary {geom} {interp} {nx}", flush=True)
    phm, scan = _scan(oracle_lib, geom, nDet, 1)
    b = _plan(gpu_ctx, geom, nDet, 1, nx, nx, interp, _info(geom, nDet, 1))
    row = np.random.default_rng(nx).standard_normal((1, nDet))
    seen = 0
    for k in range(8):  # a view at a time (a pixel that is no number stays so), some after whole turns
        angle = np.array([(k + 8 * (k % 4)) * (np.pi / 4)])
        for off in (-3, -2, -1, 0, 1, 2, 3):
            bad = row.copy()
            bad[0, (nDet - 1) // 2 + off] = np.nan
            want = oracle_lib.backproject("oracle", phm, scan, "idiff", interp, nx, nx, bad, angle)
            img = torch.zeros((nx, nx), dtype=torch.float32, device="cuda")
            b.backproject(torch.from_numpy(bad).cuda(), angle, img, ctsim_amd.PREC_F64)
            b.postprocess(img)
            torch.cuda.synchronize()
            out, nan = img.cpu().numpy(), np.isnan(want)
            seen += int(nan.sum())
            assert np.array_equal(nan, np.isnan(out)), f"view {k} cell {off}: {int((nan != np.isnan(out)).sum())} pixels"
            assert np.array_equal(out[~nan].view(np.uint32), want[~nan].view(np.uint32)), f"view {k} cell {off}"
    assert seen > 0
