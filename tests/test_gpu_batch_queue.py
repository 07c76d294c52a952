"""The batch's work queues where they are uneven: fewer items than workgroups,
many more (the queue heads count on from the workgroups' ranks), slices dealt
whole beside one dealt over all XCDs, and replays (the heads start again).
Every image pixel is written once: the images start at NaN, lie within
d <= 1e-5 of the FP64 single-slice image, and repeat bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (geometry, detectors, views, image side) per slice
BATCHES = {
    "one_tiny": [("parallel", 33, 9, 24)],
    "tiny": [("equilinear", 65, 20 + k, 32) for k in range(11)],
    "one_large": [("parallel", 401, 40, 768)],
    "large_and_tiny": [("equiangular", 301, 61, 512)] + [("parallel", 65, 30 + k, 40) for k in range(9)],
}


@pytest.mark.parametrize("P,lanesY,fused,sym", [(2, 16, True, 0), (1, 8, False, 1), (4, 16, False, 0), (2, 8, False, 8)])
@pytest.mark.parametrize("name", list(BATCHES))
def test_batch_queues(gpu_ctx, name, P, lanesY, fused, sym):
    import torch
    import ctsim_amd
    from ctsim_amd import fbp
    from ctsim_amd import workloads as W
    print(f"case batch queue {name} P={P} lanesY={lanesY} fused={fused} sym={sym}", flush=True)
    specs = [W.SliceSpec(elems=W.seeded_elements(8, 0x51 + k), geometry=g, nDet=nd, nView=nv,
                         rotLen=np.pi if g == "parallel" else 2 * np.pi, filter="abs_bandlimit", method="convolution",
                         interp="linear", backproj="idiff", filterParam=-1.0, nx=n, ny=n)
             for k, (g, nd, nv, n) in enumerate(BATCHES[name])]
    sims = [fbp.simulate(gpu_ctx, s) for s in specs]
    ref = [fbp.reconstruct(gpu_ctx, s, sino, ang, info, ctsim_amd.PREC_F64) for s, (sino, ang, info) in zip(specs, sims)]
    b = ctsim_amd.Batch(gpu_ctx, [fbp.slice_desc(s, info, ang) for s, (_, ang, info) in zip(specs, sims)])
    b.set_shape(P, lanesY, 16384, fused, sym)
    images = [torch.full((s.nx, s.ny), float("nan"), dtype=torch.float32, device="cuda") for s in specs]
    first = None
    for _ in range(3):
        for i in images:
            i.fill_(float("nan"))
        b.run([x[0] for x in sims], images)
        b.status()
        for r, i in zip(ref, images):
            assert ctsim_amd.image_stats(gpu_ctx, r, i)[0] <= 1e-5
        first = first or [i.clone() for i in images]
        assert all(torch.equal(a, i) for a, i in zip(first, images))
