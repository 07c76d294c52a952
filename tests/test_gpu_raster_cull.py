"""The rasteriser's culling of elements by 8 x 8 squares: images around the
square and the 16 x 16 tile, phantoms of every element type around the 64
elements tested at a time, small elements that fall between squares and large
ones that contain many, one to three samples a side, attenuations too small
for the culling.  Bit for bit against the oracle."""
import numpy as np
import pytest

from ctsim_amd import workloads as W

pytestmark = pytest.mark.gpu


def _elements(n, seed, scale):
    rng = np.random.default_rng(seed)
    kinds = ["ellipse", "rectangle", "triangle", "sector", "segment"]
    out = []
    for k in range(n):
        u, v = scale * rng.uniform(0.02, 1.0, size=2) ** 2
        out.append((kinds[k % 5], *map(float, rng.uniform(-1, 1, size=2)), float(u), float(v),
                    float(rng.uniform(-180, 180)), float(rng.uniform(-1, 1))))
    return out


@pytest.mark.parametrize("nx,ny,ns,n,scale,atten",
                         [(2, 2, 1, 5, 1.0, 1.0), (7, 9, 3, 63, 0.3, 1.0), (8, 16, 2, 64, 1.0, 1.0),
                          (17, 33, 1, 65, 2.0, 1.0), (130, 95, 2, 129, 0.1, 1.0), (64, 200, 1, 40, 1.5, 1.0),
                          (40, 41, 2, 70, 1.0, 1e-45), (33, 64, 2, 30, 1.0, 1e-30)])
def test_raster_matches_oracle(gpu_ctx, oracle_lib, nx, ny, ns, n, scale, atten):
    import ctsim_amd
    el = [(*e[:6], e[6] * atten) for e in _elements(n, nx + n, scale) + W.mixed_elements(5)]
    print(f"case raster {nx}x{ny} samples {ns} elements {len(el)} scale {scale} attenuation {atten}", flush=True)
    img, _ = ctsim_amd.Phantom(None, el).rasterize(gpu_ctx, nx, ny, 1.0, ns)
    ref = oracle_lib.rasterize("oracle", oracle_lib.Phantom(None, el), nx, ny, 1.0, ns)
    assert np.array_equal(img.cpu().numpy().view(np.uint32), ref.view(np.uint32))
