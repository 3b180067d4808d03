"""The matrix-core backprojection (variant 4 + 64 + 2048 of dfm_radon_backward_table) at the sizes where it can go
wrong: images smaller than a tile and with remainders, one angle, remainders of a pass, many angles, orientation counts at the edges of its 64-orientation blocks, the detector smaller than the
image. Reference: the float64 pixel table of the same geometry (radon_tables, pinned to the oracle in
test_host_tables.py), summed in float64. Tolerance per pixel: the rounding of 2 n + 2 float32 operations on the sum of
the terms' magnitudes."""
import numpy as np
import pytest

from pairs import build, cfg

pytestmark = pytest.mark.gpu

MFMA = 4 + 64 + 2048
SHAPES = [(1, 1, 3, 1, 4), (7, 9, 13, 3, 60), (9, 7, 5, 5, 64), (16, 16, 19, 66, 68), (24, 8, 27, 9, 132)]


def _setup(nx, ny, my, na, K):
    import torch
    op, _, _ = build(cfg(nx=nx, ny=ny, my=my, n_omega=na, n_eta=12, angle_range=(0, 360), cor=0.3), K=K,
                     pf_mode="sparse", oracle=False)
    tab = op._tables_full
    assert tab["mfma_ok"]
    g = torch.Generator(device="cuda").manual_seed(nx + na)
    sino = torch.rand(na * my * op.K_stride, generator=g, device="cuda") - 0.3
    return op, tab, sino, g


def _terms(op, tab, sino):
    """(w, s) of both taps of every (angle, pixel), float64, s shaped (na, npix, 2, K_stride)."""
    p = tab["ptab"].cpu().numpy()
    s = sino.view(op.N_Omega, op.My, op.K_stride).cpu().numpy().astype(np.float64)
    w = p[..., 2:].copy().view(np.float32).astype(np.float64)
    bins = np.stack([s[a][p[a, :, :2]] for a in range(op.N_Omega)])
    return w, bins


def _image(op, sino):
    import torch
    op.radon_variant.update(bwd_kernel="table", bwd=MFMA)
    img = torch.full((op.Nx * op.Ny * op.K_stride,), 7.0, device="cuda")
    op._radon_backward(sino, op.geo_bwd, op._tables_full, op.N_Omega, img, op.K_stride, 0, op.K_stride)
    torch.cuda.synchronize()
    return img.view(-1, op.K_stride).cpu().numpy()


@pytest.mark.parametrize("shape", SHAPES)
def test_sums_match_table(shape):
    print(f"case backprojection mfma {shape}", flush=True)
    op, tab, sino, _ = _setup(*shape)
    w, s = _terms(op, tab, sino)
    ref = np.einsum("apt,aptk->pk", w, s)
    tol = (2 * op.N_Omega + 2) * 2.0 ** -24 * np.einsum("apt,aptk->pk", np.abs(w), np.abs(s)) + 1e-30
    assert np.all(np.abs(_image(op, sino) - ref) <= tol)


def test_updates():
    """Modes 1 to 3 on the sums of mode 0 (their arithmetic in float32; a fused multiply-add may round once less, so
    4 roundings of the largest operand)."""
    import torch
    print(f"case backprojection mfma updates", flush=True)
    op, tab, sino, g = _setup(17, 10, 21, 11, 70)
    dz = _image(op, sino)
    n = dz.size
    r = lambda: torch.rand(n, generator=g, device="cuda")
    x0, z0 = r(), r() - 0.5
    T = r() * (r() > 0.2)
    h = lambda t: t.view(-1, op.K_stride).cpu().numpy()
    for mode, kw in (("spdhg", {}), ("em", {"em": True}), ("pdhg", {"pdhg": True})):
        x, z = x0.clone(), z0.clone()
        op._radon_backward(sino, op.geo_bwd, tab, op.N_Omega, None, op.K_stride, 0, op.K_stride, x=x, z=z, T=T,
                           inv_p=0.7, lam=0.05, **kw)
        torch.cuda.synchronize()
        f = np.float32
        X, Z, t = h(x0), h(z0), h(T)
        if mode == "spdhg":
            zn = Z + dz
            xn = np.where(t > 0, np.maximum(0, X - t * ((zn + f(0.7) * dz) + f(0.05))), 0)
        elif mode == "em":
            xn, zn = np.where(t > 0, X * dz / (t + f(0.05)), X), Z
        else:
            xn = np.where(t > 0, np.maximum(0, X - t * (dz + f(0.05))), 0)
            zn = 2 * xn - X
        for got, ref in ((h(x), xn), (h(z), zn)):
            tol = 4 * 2.0 ** -24 * max(np.abs(ref).max(), np.abs(dz).max(), 1.0)
            if mode == "em":
                tol = 4 * 2.0 ** -24 * np.abs(ref).max()
            assert np.abs(got - ref).max() <= tol, mode


def test_non_finite_bins_stay_on_their_pixels():
    """An infinite and a NaN bin reach exactly the pixels that have a weight on them."""
    print("case backprojection mfma non-finite", flush=True)
    op, tab, sino, _ = _setup(20, 17, 23, 7, 40)
    v = sino.view(op.N_Omega, op.My, op.K_stride)
    v[2, 9, 5] = float("inf")
    v[5, 11, 33] = float("nan")
    w, s = _terms(op, tab, sino)
    got = _image(op, sino)
    with np.errstate(invalid="ignore"):
        ref = np.where(w[..., None] != 0, w[..., None] * s, 0.0).sum(axis=(0, 2))
    assert np.array_equal(np.isfinite(got), np.isfinite(ref)) and np.array_equal(np.isnan(got), np.isnan(ref))
    ok = np.isfinite(ref)
    assert np.abs(got[ok] - ref[ok]).max() < 1e-5
