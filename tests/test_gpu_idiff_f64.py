"""The FP64 IntDiff backprojection with linear and cubic interpolation
(backproject_f64.hip) where its dispatch and tiles end: images around the 16-
and 32-pixel tiles and around the size from which a lane takes four rows, view
counts around the views staged at a time (16, and fewer for long windows) and
the 128 whose windows are found together, windows staged by 32 lanes, by 64
and in several rounds, detectors that end inside the image, and rows of
zeros, infinities and no numbers.  Every comparison is bit for bit."""
import numpy as np
import pytest

from conftest import record_parity
from ctsim_amd import workloads as W

pytestmark = pytest.mark.gpu


def _run(ctx, O, nx, ny, nDet, nView, interp, rows, scanRatio=1.0):
    import torch
    import ctsim_amd
    phm_o = O.Phantom(None, W.mixed_elements(31))
    scan = O.ScanSpec("parallel", nDet, nView, 0, 1, np.pi, 2.0, 2.0, 1.0, scanRatio)
    angles = np.arange(nView) * (np.pi / nView)
    want = O.backproject("oracle", phm_o, scan, "idiff", interp, nx, ny, rows, angles)
    sc = ctsim_amd.Scanner(ctsim_amd.Phantom(None, W.mixed_elements(31)), "parallel", nDet, nView, 0, 1, np.pi, 2.0,
                           2.0, 1.0, scanRatio)
    b = ctsim_amd.Backprojector(ctx, "parallel", nDet, sc.info["detInc"], nView, sc.info["viewDiameter"],
                                sc.info["focalLength"], sc.info["sourceDetectorLength"], "idiff", interp, nx, ny)
    img = torch.zeros((nx, ny), dtype=torch.float32, device="cuda")
    b.backproject(torch.from_numpy(rows).cuda(), angles, img, ctsim_amd.PREC_F64)
    b.postprocess(img)
    torch.cuda.synchronize()
    return img.cpu().numpy(), want


@pytest.mark.parametrize("interp", ["linear", "cubic"])
@pytest.mark.parametrize("nx,ny,nDet,nView,scanRatio",
                         [(16, 16, 24, 1, 1.0), (17, 33, 40, 15, 1.0), (1, 40, 65, 16, 1.0), (95, 64, 130, 17, 1.0),
                          (130, 131, 367, 130, 1.0), (40, 40, 400, 9, 1.0), (24, 30, 1500, 5, 1.0),
                          (64, 50, 97, 33, 0.5), (1025, 1030, 700, 5, 1.0), (1024, 1024, 2000, 19, 0.6)])
def test_noise_rows_match_oracle(gpu_ctx, oracle_lib, nx, ny, nDet, nView, scanRatio, interp):
    print(f"case idiff f64 {interp} {nx}x{ny} {nDet}x{nView} scan ratio {scanRatio}", flush=True)
    rows = np.random.default_rng(nx + nView).standard_normal((nView, nDet))
    out, want = _run(gpu_ctx, oracle_lib, nx, ny, nDet, nView, interp, rows, scanRatio)
    assert record_parity(f"oracle idiff f64 {interp} {nx}x{ny} {nDet}x{nView} {scanRatio}", out, want) == 0


@pytest.mark.parametrize("interp", ["linear", "cubic"])
@pytest.mark.parametrize("value", [np.inf, np.nan, 1e-60])
def test_special_rows_match_oracle(gpu_ctx, oracle_lib, interp, value):
    """One special cell in each row, beside others and at the last cell."""
    nx, ny, nDet, nView = 37, 50, 41, 6
    print(f"case idiff f64 special {interp} {value}", flush=True)
    rows = np.random.default_rng(3).standard_normal((nView, nDet)) * (1.0 if value != 1e-60 else 1e-60)
    rows[np.arange(nView), [3, 11, 20, 21, 33, 40]] = value
    out, want = _run(gpu_ctx, oracle_lib, nx, ny, nDet, nView, interp, rows)
    nan = np.isnan(want)
    assert np.array_equal(nan, np.isnan(out))
    assert np.array_equal(out[~nan].view(np.uint32), want[~nan].view(np.uint32))


@pytest.mark.parametrize("interp", ["linear", "cubic"])
def test_zeros_onto_negative_zeros(gpu_ctx, interp):
    """Zero rows of a detector that ends inside the image, onto an image of
    -0.0: linear interpolation leaves a pixel outside the detector alone,
    cubic interpolation adds +0.0 to it, as the reference does."""
    import torch
    import ctsim_amd
    nx, nDet = 40, 21
    print(f"case idiff f64 zeros {interp}", flush=True)
    b = ctsim_amd.Backprojector(gpu_ctx, "parallel", nDet, 0.05, 1, 2.0 * np.sqrt(2.0), 2.0, 4.0, "idiff", interp, nx, nx)
    img = torch.full((nx, nx), -0.0, dtype=torch.float32, device="cuda")
    b.backproject(torch.zeros((1, nDet), dtype=torch.float64, device="cuda"), np.zeros(1), img, ctsim_amd.PREC_F64)
    torch.cuda.synchronize()
    # at angle 0 the position is 10 + x / 0.05, x = -1 + 0.05 (ix + 0.5) to a rounding: cells [0, 21) are ix 10 ... 30,
    # the first of them half a cell in
    sign = np.signbit(img.cpu().numpy())
    inside = np.arange(nx)
    inside = (inside >= 10) & (inside <= 30)
    assert np.array_equal(sign[inside], np.zeros((21, nx), bool))
    assert np.array_equal(sign[~inside], np.full((nx - 21, nx), interp == "linear"))
