"""The FP64 ray sums' short chords (ellipses and rectangles) where they must
hand over to the reference's chain: rays that graze an ellipse or run along a
rectangle's side or through its corners, needles and large aspects, elements
that reach beyond the source or the detector, elements whose chords cancel,
phantoms with other types among them, detector counts around the 64 of a wave,
two and three samples per detector, and scans of one view.  Bit for bit against
the oracle."""
import numpy as np
import pytest

from conftest import record_parity
from ctsim_amd import workloads as W

pytestmark = pytest.mark.gpu


def _ellipses(n, seed, lo, hi):
    rng = np.random.default_rng(seed)
    return [("ellipse", *map(float, rng.uniform(-0.7, 0.7, 2)), *map(float, rng.uniform(lo, hi, 2)),
             float(rng.uniform(0, 180)), float(rng.uniform(-1, 1))) for _ in range(n)]


BOX = [("rectangle", 0.0, 0.0, 1.0, 1.0, 0.0, 0.1)]
PHANTOMS = {
    # concentric circles, whose tangents the detector grid meets again and again
    "circles": BOX + [("ellipse", 0.0, 0.0, r, r, 0.0, 0.3) for r in np.linspace(0.05, 0.95, 19)],
    "squares": BOX + [("rectangle", x, y, 0.1, 0.1, 0.0, 0.2) for x in (-0.5, 0.0, 0.5) for y in (-0.5, 0.0, 0.5)],
    "turned": BOX + [("rectangle", 0.1 * k, -0.05 * k, 0.3, 0.02, 10.0 * k, 0.5) for k in range(-5, 6)],
    "needles": _ellipses(12, 4, 1e-6, 0.4) + [("ellipse", 0.0, 0.0, 1.0, 1.0, 0.0, 0.01)],
    "cancel": [e for k, e in enumerate(_ellipses(8, 5, 0.1, 0.4)) for e in (e, (*e[:6], -e[6]))] + BOX,
    "mixed": W.mixed_elements(9) + _ellipses(70, 6, 0.02, 0.3),
    "one": [("ellipse", 0.0, 0.0, 0.5, 0.25, 30.0, 1.0)],
}


@pytest.mark.parametrize("geom", ["parallel", "equiangular", "equilinear"])
@pytest.mark.parametrize("name", list(PHANTOMS))
@pytest.mark.parametrize("nDet,nView,nSample,focal", [(127, 36, 1, 2.0), (64, 8, 3, 2.0), (130, 5, 2, 1.02), (1, 1, 1, 2.0),
                                                      (65, 12, 1, 0.9)])
def test_raysums_match_oracle(gpu_ctx, oracle_lib, name, geom, nDet, nView, nSample, focal):
    import torch
    import ctsim_amd
    if focal < 1 and geom != "parallel":
        pytest.skip("a fan beam's source lies outside the scanned circle")
    print(f"case short raysum {name} {geom} {nDet}x{nView} samples {nSample} focal {focal}", flush=True)
    O, elems = oracle_lib, PHANTOMS[name]
    rot = np.pi if geom == "parallel" else 2 * np.pi
    ref = O.pipeline("oracle", O.Phantom(None, elems), O.ScanSpec(geom, nDet, nView, 0, nSample, rot, focal, focal))
    sc = ctsim_amd.Scanner(ctsim_amd.Phantom(None, elems), geom, nDet, nView, 0, nSample, rot, focal, focal)
    sino = torch.zeros((nView, nDet), dtype=torch.float32, device="cuda")
    sc.collect(gpu_ctx, sino, ctsim_amd.PREC_F64)
    torch.cuda.synchronize()
    assert record_parity(f"oracle short raysum {name} {geom} {nDet}x{nView}x{nSample} {focal}", sino.cpu().numpy(),
                         ref["sino"]) == 0


# scans large enough that items which meet another type go to the chain by themselves, and scans whose rays end
# in the disc of the elements (the detector's middle, or the rim)
FEW_OTHERS = BOX + _ellipses(20, 8, 0.02, 0.3) + [("triangle", 0.4, 0.1, 0.03, 0.05, 20.0, 0.4)]


@pytest.mark.parametrize("name,geom,nDet,nView,focal,center", [
    ("others", "parallel", 130, 1100, 2.0, 2.0), ("others", "equiangular", 200, 800, 2.0, 2.0),
    ("others", "equilinear", 191, 1030, 2.0, 2.0), ("circles", "parallel", 127, 40, 1.0, 1.0),
    ("turned", "parallel", 200, 33, 2.0, 1.0), ("circles", "equilinear", 130, 40, 2.0, 1.0),
    ("turned", "equilinear", 130, 40, 2.0, 0.9), ("circles", "equiangular", 130, 40, 2.0, 1.0)])
def test_deferred_items_match_oracle(gpu_ctx, oracle_lib, name, geom, nDet, nView, focal, center):
    import torch
    import ctsim_amd
    print(f"case short raysum {name} {geom} {nDet}x{nView} focal {focal} center {center}", flush=True)
    O, elems = oracle_lib, FEW_OTHERS if name == "others" else PHANTOMS[name]
    rot = np.pi if geom == "parallel" else 2 * np.pi
    ref = O.pipeline("oracle", O.Phantom(None, elems), O.ScanSpec(geom, nDet, nView, 0, 1, rot, focal, center))
    sc = ctsim_amd.Scanner(ctsim_amd.Phantom(None, elems), geom, nDet, nView, 0, 1, rot, focal, center)
    sino = torch.zeros((nView, nDet), dtype=torch.float32, device="cuda")
    sc.collect(gpu_ctx, sino, ctsim_amd.PREC_F64)
    torch.cuda.synchronize()
    assert record_parity(f"oracle short raysum {name} {geom} {nDet}x{nView} {focal} {center}", sino.cpu().numpy(),
                         ref["sino"]) == 0
