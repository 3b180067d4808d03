"""The line-sweep forward projection (dfm_radon_forward_lines) at the sizes where it can go wrong: lines shorter than one
load instruction, at its edges and up to 256 pixels, both layouts, more line ranges than lines, orientation counts that
leave a part of a block, both sweep classes. Reference: the float64 geometry table (radon_tables, pinned to the oracle in
test_host_tables.py) summed in float64. Tolerance per ray: the rounding of 6 float32 operations per line on the terms'
magnitudes, and 8 units of rounding in each of the 3 weights per line (a weight is formed from terms of at most 4)."""
import numpy as np
import pytest

from pairs import build, cfg

pytestmark = pytest.mark.gpu


def _setup(nx, ny, my, na, K):
    import torch
    op, _, _ = build(cfg(nx=nx, ny=ny, my=my, n_omega=na, n_eta=12, angle_range=(0, 360), cor=0.3), K=K,
                     pf_mode="sparse", oracle=False)
    assert op._tables_full["pairs_ok"]
    g = torch.Generator(device="cuda").manual_seed(nx + na)
    return op, torch.rand(nx * ny * op.K_stride, generator=g, device="cuda") - 0.3


def _sino(op, img, nsplit, dup):
    import torch
    op.radon_variant.update(fwd_kernel="lines", fwd_lines=nsplit + 128 * dup)
    s = torch.full((op.N_Omega * op.My * op.K_stride,), 7.0, device="cuda")
    op._radon_forward(img, op.K_stride, 0, op.K_stride, s, op.geo_fwd, op.N_Omega, op._tables_full)
    torch.cuda.synchronize()
    return s.view(-1, op.K_stride).cpu().numpy()


def _reference(op, img):
    """(sums, sums of magnitudes) per (ray, orientation) from the table, float64."""
    t = {k: op._tables_full[k].cpu().numpy() for k in ("row_ptr", "pix", "w")}
    x = img.view(-1, op.K_stride).cpu().numpy().astype(np.float64)
    n = op.N_Omega * op.My
    ref, mag = np.zeros((n, op.K_stride)), np.zeros((n, op.K_stride))
    for r in range(n):
        e = slice(t["row_ptr"][r], t["row_ptr"][r + 1])
        w, v = t["w"][e].astype(np.float64)[:, None], x[t["pix"][e]]
        with np.errstate(invalid="ignore"):
            ref[r], mag[r] = (w * v).sum(0), np.abs(w * v).sum(0)
    return ref, mag


@pytest.mark.parametrize("shape", [(1, 1, 3, 2, 4), (9, 3, 13, 6, 33), (32, 31, 35, 7, 64), (65, 64, 70, 12, 70),
                                   (128, 3, 131, 4, 20), (200, 9, 205, 5, 12), (256, 16, 259, 3, 8)])
def test_sums_match_table(shape):
    print(f"case lines {shape}", flush=True)
    op, img = _setup(*shape)
    ref, mag = _reference(op, img)
    n = max(op.Nx, op.Ny)
    scale = float(op.radon_scale) * float(np.max(op._geo64["inv_a"]))
    tol = (6 * n + 2) * 2.0 ** -24 * mag + 3 * n * 8 * 2.0 ** -24 * scale * float(img.abs().max())
    forms = [(1, 0), (1, 1), (2, 1), (5, 0), (64, 1)]
    got = {f: _sino(op, img, *f) for f in forms}
    for f in forms:
        assert np.all(np.abs(got[f] - ref) <= tol), f
    assert np.array_equal(got[1, 0], got[1, 1])


def test_equals_register_staged_sweep():
    import torch
    print("case lines against psweep", flush=True)
    op, img = _setup(99, 99, 103, 9, 100)
    got = _sino(op, img, 1, 1)
    op.radon_variant.update(fwd_kernel="psweep", fwd_psweep=2)
    s = torch.empty(op.N_Omega * op.My * op.K_stride, device="cuda")
    op._radon_forward(img, op.K_stride, 0, op.K_stride, s, op.geo_fwd, op.N_Omega, op._tables_full)
    torch.cuda.synchronize()
    assert np.array_equal(got, s.view(-1, op.K_stride).cpu().numpy())


def test_non_finite_pixels_stay_on_their_rays():
    """An infinite and a NaN pixel reach exactly the rays that have a weight on them."""
    print("case lines non-finite", flush=True)
    op, img = _setup(30, 23, 33, 8, 40)
    v = img.view(23, 30, op.K_stride)
    v[11, 14, 5] = float("inf")
    v[7, 20, 33] = float("nan")
    ref, _ = _reference(op, img)
    for f in ((1, 0), (1, 1), (3, 1)):
        got = _sino(op, img, *f)
        assert np.array_equal(np.isfinite(got), np.isfinite(ref)) and np.array_equal(np.isnan(got), np.isnan(ref))
        ok = np.isfinite(ref)
        assert np.abs(got[ok] - ref[ok]).max() < 1e-4


@pytest.mark.parametrize("K", [12, 200])
def test_subsets_of_different_sizes_under_graphs(K):
    """Steps of subsets of 3 and 4 angles replayed from graphs equal eager steps (the partial-sum workspace serves the
    largest subset)."""
    import torch
    from diffractom_amd import SPDHGPoisson
    print(f"case lines graphs K={K}", flush=True)
    c = cfg(nx=70, ny=68, my=73, n_omega=11, n_eta=12)
    out = []
    for graphs in (False, True):
        op, _, _ = build(c, K=K, pf_mode="sparse", pf_precision="bf16_residual", oracle=False)
        b = torch.poisson(torch.full(op.data_shape, 20.0), generator=torch.Generator().manual_seed(1)).cuda()
        sol = SPDHGPoisson(op, subsets=3, seed=0)
        sol.graphs = graphs
        sol.start(torch.zeros(op.coeff_shape, device="cuda"), b)
        sol.advance(5)
        torch.cuda.synchronize()
        sol.advance(7)
        torch.cuda.synchronize()
        out.append(sol.xk.cpu().numpy())
    assert np.array_equal(out[0], out[1])


def test_workspace_belongs_to_the_operators_stream():
    """The partial sums' workspaces of an operator with a stream of its own come from that stream's memory, and its
    products equal those on the current stream."""
    import torch
    print("case lines workspace stream", flush=True)
    out = []
    for queue in (None, torch.cuda.Stream()):
        op, _, _ = build(cfg(nx=84, ny=83, my=87, n_omega=12, n_eta=36), K=800, pf_mode="sparse",
                         pf_precision="bf16_residual", oracle=False)
        op.queue = queue
        x = torch.rand(op.coeff_shape, generator=torch.Generator().manual_seed(3)).cuda()
        d = torch.zeros(op.data_shape, device="cuda")
        torch.cuda.synchronize()
        op.direct_cl(x, d)
        torch.cuda.synchronize()
        out.append(d.cpu().numpy())
        for buf in (op._t_buf_t, op._mfma_part_buf):
            seg = [s for s in torch.cuda.memory_snapshot() if s["address"] <= buf.data_ptr() < s["address"] + s["total_size"]]
            assert len(seg) == 1 and seg[0]["stream"] == (0 if queue is None else queue.cuda_stream)
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("koff,kn", [(0, 4), (8, 20), (32, 32), (12, 52)])
def test_column_ranges(koff, kn):
    """Column ranges that fill a part of a block of 32 orientations: the columns of the whole product, nothing beyond."""
    import torch
    from diffractom_amd import _lib
    print(f"case lines columns koff={koff} kn={kn}", flush=True)
    op, img = _setup(40, 33, 43, 7, 64)
    whole = _sino(op, img, 1, 1)
    t, g = op._tables_full, op._tables_full["sweep_grp_p"]
    for nsplit, dup in ((1, 1), (3, 0)):
        out = torch.full((op.N_Omega * op.My, 64), 7.0, device="cuda")
        part = torch.empty(nsplit * out.numel(), device="cuda")
        _lib.call("dfm_radon_forward_lines", _lib.ptr(img), _lib.ptr(out), _lib.ptr(part), _lib.ptr(t["sweep_geo"]),
                  _lib.ptr(g), _lib.ptr(t["sweep_gcls_p"]), g.shape[0], g.shape[1], op.N_Omega, op.My, op.Nx, op.Ny,
                  op.K_stride, koff, kn, 64, nsplit, dup, op._stream())
        got = out.cpu().numpy()
        assert np.all(got[:, kn:] == 7.0)
        ref = whole[:, koff:koff + kn]
        # split lines: the sums' order differs, 6 roundings per line on terms of one magnitude
        tol = 0.0 if nsplit == 1 else (6 * 40 + 2) * 2.0 ** -24 * float(img.abs().max()) * 40 * 4 * op.radon_scale
        assert np.abs(got[:, :kn] - ref).max() <= tol
