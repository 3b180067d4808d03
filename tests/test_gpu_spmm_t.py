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


def _split_rule(my, n_seg, n_ang, kb):
    from diffractom_amd.operator import SinglePhaseForwardOperator
    op = object.__new__(SinglePhaseForwardOperator)
    op.My, op.N_seg, op.csr_variant = my, n_seg, {}
    return op._tsplit(n_ang, kb)


@pytest.mark.parametrize("my", [60, 103, 131, 200])
@pytest.mark.parametrize("n_ang,ncols,fill", [(18, 1500, 0.06), (9, 5000, 0.06), (23, 543, 0.2), (120, 700, 0.1)])
def test_split_forward_error_against_64_bits(n_ang, ncols, fill, my):
    """The forward's orientation sums, split by the operator's rule, are no further from the products in float64 than
    those of the finest split (ranges of 128 orientations or more, up to 1024 workgroups of 256 rows), in root mean
    square, each summed as one FP32 chain per range and the ranges in order (formed here on the CPU). Bound 1.25: 1.1 for
    the rule, the rest for two samples' difference."""
    import torch
    print(f"case spmm_t error my={my} n_ang={n_ang} ncols={ncols}", flush=True)
    rng = np.random.default_rng(my + ncols)
    n_seg, stored = 900, 2                                   # the angles repeat two stored ones
    keep = rng.random((stored, n_seg, ncols)) < fill
    pf = np.where(keep, rng.random(keep.shape) ** 2, 0.0).astype(np.float32)
    rp = np.concatenate([[0], np.cumsum(keep.sum(axis=2).ravel())]).astype(np.int32)
    dev = lambda v: torch.from_numpy(v).cuda()
    rp_d, col_d, val_d = dev(rp), dev(np.nonzero(keep)[2].astype(np.uint16).view(np.int16)), dev(pf[keep])
    ys, ld = -(-my // 4) * 4, -(-ncols // 4) * 4
    x = rng.random((stored, my, ld)).astype(np.float32)
    om = dev((np.arange(n_ang) % stored).astype(np.int32))
    xs = dev(x)[om.long()].contiguous()
    ns, st = _split_rule(my, n_seg, n_ang, ncols), _lib.stream_handle()
    out = torch.empty((ns, n_ang, n_seg, ys), device="cuda")
    _lib.call("dfm_spmm_t_direct", _lib.ptr(xs), ld, ys, _lib.ptr(rp_d), _lib.ptr(col_d), _lib.ptr(val_d),
              _lib.ptr(out), 0, ys, _lib.ptr(om), n_ang, my, ncols, n_seg, n_seg, 0, 1.0, ns, 0, st)
    got = out[:, :stored, :, :my].cpu().numpy()
    tot = got[0]
    for part in got[1:]:
        tot = tot + part
    yy = np.linspace(0, my - 1, min(my, 12)).astype(int)     # a part of the positions on the CPU
    x64, p64 = x[:, yy, :ncols].astype(np.float64), pf.astype(np.float64)
    ref = np.einsum("arc,ayc->ary", p64, x64)
    rows = 256 if my <= 128 else 128
    fine = max(1, min(64, -(-1024 // (-(-n_seg // rows) * n_ang)), ncols // 128))
    span = (-(-ncols // fine) + 3) // 4 * 4
    chain = np.zeros(ref.shape, np.float32)
    for lo in range(0, ncols, span):
        acc = np.zeros(ref.shape, np.float32)
        for c in range(lo, min(lo + span, ncols)):
            acc = (acc + p64[:, :, c, None] * x64[:, None, :, c]).astype(np.float32)
        chain += acc
    rms = lambda v: np.sqrt(np.mean((v - ref) ** 2))
    assert rms(tot[:, :, yy]) <= 1.25 * rms(chain), (rms(tot[:, :, yy]), rms(chain), ns, fine)
