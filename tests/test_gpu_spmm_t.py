"""The CSR products on transposed operands at the edges of their tiles: every block count of 64 detector positions with a
remainder and without, workgroups of 4, 2 and 1 row quads per wave (by the launch's size), rows without entries, rows of
more entries than the two windows loaded ahead, columns that end inside a staging quad, column splits, both operand
forms and both output forms. Against the products in float64 (pf_kernels.cl:597-687)."""
import numpy as np
import pytest

from diffractom_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_ang", [32, 22, 3])               # 4, 2 and 1 row quads (2, 2 and 1 above 128 positions)
@pytest.mark.parametrize("my", [1, 16, 63, 64, 65, 103, 128, 129, 200, 257, 321, 385, 449, 512])
def test_products_at_tile_edges(my, n_ang):
    import torch
    print(f"case spmm_t my={my} n_ang={n_ang}", flush=True)
    rng = np.random.default_rng(my)
    nrows, ncols, rows_out = 299, 333, 304
    keep = rng.random((n_ang, nrows, ncols)) < 0.06
    keep[0] = False                                          # an angle without entries
    keep[1, 7] = keep[1, 130] = True                         # full rows beside sparse ones
    keep[:, 5] = False
    pf = np.where(keep, rng.random(keep.shape) - 0.3, 0.0).astype(np.float32)
    rp = np.concatenate([[0], np.cumsum(keep.sum(axis=2).ravel())]).astype(np.int32)
    col = np.nonzero(keep)[2].astype(np.uint16)
    dev = lambda v: torch.from_numpy(v).cuda()
    rp_d, col_d, val_d = dev(rp), dev(col.view(np.int16)), dev(pf[keep])
    ys, ld, old = -(-my // 4) * 4, 336, 308
    x = (rng.random((n_ang, my, ld)) - 0.3).astype(np.float32)
    xt = np.full((n_ang, ncols, ys), np.nan, np.float32)     # the padding is never part of a result
    xt[:, :, :my] = x[:, :, :ncols].transpose(0, 2, 1)
    om = np.arange(n_ang, dtype=np.int32)[::-1].copy()
    om_d, st = dev(om), _lib.stream_handle()
    p64, x64 = pf[om].astype(np.float64), x[:, :, :ncols].astype(np.float64).transpose(0, 2, 1)
    ref, mag = p64 @ x64, np.abs(p64) @ np.abs(x64)          # (a, row, y)
    rel = (ncols + 4) * 2.0 ** -24                           # a chain of at most ncols FMAs, the splits' sum, alpha
    for src, in_ld in ((dev(x), ld), (dev(xt), 0)):
        for nsplit, kc in ((2, 0), (2, 24)):
            out = torch.full((nsplit, n_ang, rows_out, ys), 7.0, device="cuda")
            _lib.call("dfm_spmm_t_direct", _lib.ptr(src), in_ld, ys, _lib.ptr(rp_d), _lib.ptr(col_d), _lib.ptr(val_d),
                      _lib.ptr(out), 0, ys, _lib.ptr(om_d), n_ang, my, ncols, nrows, rows_out, 0, 1.0, nsplit, kc, st)
            got = out.cpu().numpy().astype(np.float64)
            assert np.all(got[..., my:] == 7.0)
            got = got[..., :my].sum(axis=0)
            assert np.all(np.abs(got[:, :nrows] - ref) <= rel * mag) and np.all(got[:, nrows:] == 0.0)
        out = torch.full((n_ang, my, old), 7.0, device="cuda")
        _lib.call("dfm_spmm_t_direct", _lib.ptr(src), in_ld, ys, _lib.ptr(rp_d), _lib.ptr(col_d), _lib.ptr(val_d),
                  _lib.ptr(out), old, 0, _lib.ptr(om_d), n_ang, my, ncols, nrows, rows_out, 0, 2.0, 1, 0, st)
        got = out.cpu().numpy().astype(np.float64).transpose(0, 2, 1)
        assert np.all(np.abs(got[:, :nrows] - 2.0 * ref) <= 2.0 * rel * mag)
        assert np.all(got[:, nrows:rows_out] == 0.0) and np.all(got[:, rows_out:] == 7.0)
