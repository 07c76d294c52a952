"""Positions of the plain and mirror equilinear kernels at the fast precision:
no further from 64 bits than FP32 arithmetic on the pixels' own coordinates,
which at these sizes (short binary fractions) carry no rounding that a scaled
coordinate would add.  The same sums are formed on the CPU with every FP32
operation of

    rc = y sin + x cos,  fl = F + x sin - y cos,  q = 1 / fl,
    position = (rc q) (SDL / increment) + centre - window start,  weight = (F q)^2

on cosine, sine and F rounded to FP32, and with all of it in FP64.  The
kernel's own reciprocal is within an ulp where the CPU's is within a half, for
which a twentieth is allowed in norm."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

f4, f8 = np.float32, np.float64


def _fma(a, b, c):
    return (a.astype(f8) * b + c).astype(f4)


def _image(rows, angles, nx, nDet, F, sdl, inc, fast):
    """Sum over the views of weight times the line through two cells; fast: by
    the FP32 operations above, windows per 16 x 16 pixels."""
    half = 1.0
    c = -half + (np.arange(nx) + 0.5) * (2 * half / nx)
    X, Y = np.meshgrid(c, c, indexing="ij")
    center = (nDet - 1) // 2
    img = np.zeros((nx, nx))
    for row, th in zip(rows, angles):
        co, si = np.cos(th), np.sin(th)
        pos = (Y * si + X * co) / (F + X * si - Y * co) * (sdl / inc) + center
        if fast:
            lo = np.floor(pos.reshape(nx // 16, 16, nx // 16, 16).min(axis=(1, 3))) - 2
            lo = np.kron(lo, np.ones((16, 16)))
            x, y, co, si = X.astype(f4), Y.astype(f4), f4(co), f4(si)
            rc, fl = _fma(y, f8(si), x * co), _fma(-y, f8(co), _fma(x, f8(si), f8(f4(F))))
            q = (1 / fl.astype(f8)).astype(f4)
            rel = _fma(rc * q, f8(f4(sdl / inc)), center - lo)
            cell, u = np.floor(rel), rel - np.floor(rel)
            i = (cell + lo).astype(int)
            w = (f4(F) * q) * (f4(F) * q)
        else:
            cell = np.floor(pos)
            i, u = cell.astype(int), pos - cell
            w = (F / (F + X * si - Y * co)) ** 2
        ok = (i >= 0) & (i < nDet - 1)
        i = np.clip(i, 0, nDet - 2)
        if fast:
            d = row[1:] - row[:-1]
            v = _fma(u, d[i].astype(f8), row[i].astype(f8)).astype(f8) * w
        else:
            r = row.astype(f8)
            v = (r[i] + u * (r[i + 1] - r[i])) * w
        img += np.where(ok, v, 0.0)
    return img


@pytest.mark.parametrize("sym", [0, 3])
@pytest.mark.parametrize("nDet,nView,nx", [(183, 90, 128), (1413, 582, 128), (500, 1300, 256)])
def test_positions_keep_their_precision(gpu_ctx, nDet, nView, nx, sym):
    import torch
    import ctsim_amd
    print(f"case equilinear precision {nDet}x{nView} {nx}^2 sym={sym}", flush=True)
    d = 2 * np.sqrt(2.0)
    F, sdl = d, 2 * d
    inc = 2 * sdl * np.tan(np.arcsin(0.5)) / nDet
    angles = np.arange(nView) * (2 * np.pi / nView)
    rows = np.random.default_rng(nDet).standard_normal((nView, nDet)).astype(f4)
    rows = (rows + np.roll(rows, 1, 1) + np.roll(rows, 2, 1)).astype(f4)  # a signal wider than a cell
    exact = _image(rows, angles, nx, nDet, F, sdl, inc, False)
    limit = np.linalg.norm(_image(rows, angles, nx, nDet, F, sdl, inc, True) - exact)
    bp = ctsim_amd.Backprojector(gpu_ctx, "equilinear", nDet, inc, nView, d, F, sdl, "idiff", "linear", nx, nx)
    bp.set_shape(16, 1, 8, 4, sym)
    img = torch.zeros((nx, nx), dtype=torch.float32, device="cuda")
    bp.backproject(torch.from_numpy(rows).cuda(), angles, img, ctsim_amd.PREC_MIXED)
    torch.cuda.synchronize()
    err = np.linalg.norm(img.cpu().numpy().astype(f8) - exact)
    print(f"  error {err / np.linalg.norm(exact):.3e}, FP32 on unscaled coordinates {limit / np.linalg.norm(exact):.3e}")
    assert err <= 1.05 * limit
