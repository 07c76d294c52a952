"""The FP64 convolution at the ends of its blocks: detector counts around the
outputs of a wave and a block and the 64 cells staged at a time, view counts
around the 64 of a wave, with 2, 4 and 8 outputs per wave (the largest that
gives every CU a block), with and without fan-beam weights, up to the largest
detector count it takes.  Bit for bit against the oracle, whose sums run in
the reference's order."""
import numpy as np
import pytest

from conftest import record_parity

pytestmark = pytest.mark.gpu


def _both(ctx, O, n, nView, geom):
    import torch
    import ctsim_amd
    sig = np.random.default_rng(n + nView).standard_normal((nView, n)).astype(np.float32)
    sig[:, : n // 5] = 0.0
    ps = ctsim_amd.ProcessSignal(ctx, "abs_hanning", "convolution", 1 / 0.002, 0.002, n, geometry=geom,
                                 focalLength=2.1, sourceDetectorLength=4.2)
    out = torch.zeros((nView, n), dtype=torch.float64, device="cuda")
    ps.filter(torch.from_numpy(sig).cuda(), out, ctsim_amd.PREC_F64)
    torch.cuda.synchronize()
    ref, _, _ = O.filter_views("oracle", sig, "abs_hanning", "convolution", bw=1 / 0.002, inc=0.002, geometry=geom,
                               focal=2.1, sdl=4.2)
    return out.cpu().numpy(), ref


# two outputs per wave but for the last two shapes (4 and 8)
@pytest.mark.parametrize("geom", [0, 1, 2])
@pytest.mark.parametrize("n,nView", [(2, 1), (7, 3), (8, 64), (9, 65), (64, 63), (65, 128), (128, 70), (367, 130),
                                     (700, 500), (1030, 500)])
def test_convolution_matches_oracle(gpu_ctx, oracle_lib, n, nView, geom):
    print(f"case conv f64 {n}x{nView} geometry {geom}", flush=True)
    out, ref = _both(gpu_ctx, oracle_lib, n, nView, geom)
    assert record_parity(f"oracle conv f64 {n}x{nView} {geom}", out, ref) == 0


def test_largest_detector_count(gpu_ctx, oracle_lib):
    import ctsim_amd
    print("case conv f64 4033", flush=True)
    out, ref = _both(gpu_ctx, oracle_lib, 4033, 3, 0)
    assert record_parity("oracle conv f64 4033x3 0", out, ref) == 0
    with pytest.raises(ctsim_amd.CtsimError):
        _both(gpu_ctx, oracle_lib, 4034, 3, 0)
