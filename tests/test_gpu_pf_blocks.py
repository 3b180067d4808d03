"""The block-sparse PF products at the edges of their tiles: detector rows at every y-tile count and in two groups, a
contraction shorter than one chunk of 32 and one with a remainder, unaligned segment counts, blocks of more entries
than the prefetched 256 and blocks without any, a k split. Against the products in float64 (pf_kernels.cl:597-687)."""
import numpy as np
import pytest

from diffractom_amd import _lib

pytestmark = pytest.mark.gpu

MODES = {"bf16": 0, "bf16_residual": 1, "fp16": 2}


def _store(dense, precision, P):
    """The block lists of a dense (R, K, CP) PF and 1 / ring scale."""
    import torch
    R, K, CP = dense.shape
    n_kb, n_jb = -(-K // 32), -(-CP // 32)
    st = _lib.stream_handle()
    cnt = torch.empty(R * n_kb * n_jb, dtype=torch.int32, device="cuda")
    _lib.call("dfm_pfblk_count", _lib.ptr(dense), _lib.ptr(cnt), R, K, K, CP, st)
    ptr = torch.zeros(cnt.numel() + 1, dtype=torch.int32, device="cuda")
    ptr[1:] = torch.cumsum(cnt, 0)
    n, f16 = int(ptr[-1]), precision == "fp16"
    pos = torch.empty(max(n, 1), dtype=torch.int16, device="cuda")
    val = torch.empty(max(n, 1), dtype=torch.int16 if f16 else torch.int32, device="cuda")
    scale = torch.full((P,), 2.0 ** 10, device="cuda") if f16 else None
    _lib.call("dfm_pfblk_fill", _lib.ptr(dense), _lib.ptr(ptr), _lib.ptr(pos), _lib.ptr(val), int(f16),
              _lib.ptr(scale), P, R, K, K, CP, st)
    return ptr, pos, val, (1.0 / scale if f16 else None), st


def _bf16(v):
    import torch
    return torch.from_numpy(np.ascontiguousarray(v)).bfloat16().float().numpy()


def _product(y, pf, precision):
    """sum_q y[a, i, q] pf[a, q, c] of the operands as the mode holds them, and the sum of magnitudes, in float64."""
    y, pf = np.asarray(y, np.float32), np.asarray(pf, np.float32)
    if precision == "fp16":
        yr = np.empty(y.shape, np.float64)
        for q in range(0, y.shape[2], 32):                   # every (row, chunk of 32): largest magnitude in 2^13 .. 2^14
            m = np.abs(y[:, :, q:q + 32]).max(axis=2, keepdims=True)
            sc = np.where(m > 0, np.ldexp(1.0, 14 - np.frexp(m)[1]), 1.0)
            yr[:, :, q:q + 32] = (y[:, :, q:q + 32] * sc).astype(np.float16).astype(np.float64) / sc
        pr = (pf * np.float32(2.0 ** 10)).astype(np.float16).astype(np.float64) / 2.0 ** 10
        return yr @ pr, np.abs(yr) @ np.abs(pr)
    yh, ph = _bf16(y), _bf16(pf)
    f = lambda v: v.astype(np.float64)
    ref = f(yh) @ f(ph)
    if precision == "bf16_residual":
        ref += f(yh) @ f(_bf16(pf - ph)) + f(_bf16(y - yh)) @ f(ph)
    return ref, np.abs(f(y)) @ np.abs(f(pf)) * (1 + 2.0 ** -6)


@pytest.mark.parametrize("precision", list(MODES))
@pytest.mark.parametrize("my,K,CP,ksplit", [(9, 20, 21, 1), (32, 70, 45, 2), (40, 33, 130, 1), (64, 130, 63, 3),
                                            (79, 97, 31, 1), (96, 64, 101, 2), (103, 200, 77, 3), (128, 31, 95, 1),
                                            (131, 161, 39, 1)])
def test_block_products_at_tile_edges(my, K, CP, ksplit, precision):
    import torch
    print(f"case pf blocks my={my} K={K} CP={CP} ksplit={ksplit} {precision}", flush=True)
    R, P = 5, 3
    rng = np.random.default_rng(my + K)
    pf = np.where(rng.random((R, K, CP)) < 0.06, rng.random((R, K, CP)), 0.0)
    pf[1] = rng.random((K, CP))                              # full blocks
    pf[2] = 0.0                                              # no entries at all
    pf[3, :, 32:] = 0.0                                      # empty blocks beside filled ones
    pf = pf.astype(np.float32)
    dense = torch.from_numpy(pf).cuda()
    ptr, pos, val, inv, st = _store(dense, precision, P)
    om = torch.tensor([4, 1, 2, 3], dtype=torch.int32, device="cuda")
    sks = (K + 3) // 4 * 4 + 4
    sino = (rng.random((4, my, sks)) - 0.3).astype(np.float32)
    data = (rng.random((R, my, CP)) - 0.3).astype(np.float32)
    # the products of the operands as the mode holds them (exact in FP32), so only the FP32 accumulation of up to three
    # products a term is left, relative to the sum of magnitudes
    rel = 3 * (max(K, CP) + 4) * 2.0 ** -23
    d_sino = torch.from_numpy(sino).cuda()
    ks = min(ksplit, -(-K // 32))
    part = torch.empty(ks * 4 * my * CP, device="cuda")
    rows = om.cpu().numpy()
    pfs, sinos, datas = pf[rows], sino[:, :, :K], data[rows]
    for waves in (0, 32):
        for acc in (0, 1):
            out = torch.from_numpy(data).cuda()
            _lib.call("dfm_pfblk_forward", _lib.ptr(d_sino), sks, K, _lib.ptr(ptr), _lib.ptr(pos), _lib.ptr(val),
                      MODES[precision] + waves, _lib.ptr(inv), P, _lib.ptr(om), 4, my, CP, _lib.ptr(out),
                      _lib.ptr(part), ks, acc, st)
            out = out.cpu().numpy()
            prev = datas.astype(np.float64) if acc else 0.0
            ref, mag = _product(sinos, pfs, precision)
            assert np.all(np.abs(out[rows] - (ref + prev)) <= rel * (mag + np.abs(prev)))
            assert np.array_equal(out[0], data[0])           # the row outside the list
        d_data = torch.from_numpy(data).cuda()
        back = torch.full((4, my, sks), np.nan, device="cuda")
        _lib.call("dfm_pfblk_adjoint", _lib.ptr(d_data), _lib.ptr(ptr), _lib.ptr(pos), _lib.ptr(val),
                  MODES[precision] + waves, _lib.ptr(inv), P, _lib.ptr(om), 4, my, CP, K, _lib.ptr(back), sks, 2.0, st)
        back = back.cpu().numpy().astype(np.float64)
        ref, mag = _product(datas, pfs.transpose(0, 2, 1), precision)
        assert np.all(np.abs(back[:, :, :K] - 2.0 * ref) <= rel * 2.0 * mag)
        assert np.all(back[:, :, K:] == 0.0)


@pytest.mark.parametrize("precision", list(MODES))
@pytest.mark.parametrize("my,K,CP", [(1, 1, 1), (17, 12, 33), (40, 33, 31), (103, 95, 70), (131, 20, 5)])
def test_values_beside_the_columns_stay_out(my, K, CP, precision):
    """NaN in the sinogram's columns beyond the orientations, in the data rows of other angles and behind the last row:
    the chunk with fewer than 32 columns takes in none of them."""
    import torch
    print(f"case pf blocks padding my={my} K={K} CP={CP} {precision}", flush=True)
    R, P = 4, 1
    rng = np.random.default_rng(my + K)
    pf = np.where(rng.random((R, K, CP)) < 0.4, rng.random((R, K, CP)), 0.0).astype(np.float32)
    ptr, pos, val, inv, st = _store(torch.from_numpy(pf).cuda(), precision, P)
    om = torch.tensor([1, 3], dtype=torch.int32, device="cuda")
    sks = (K + 3) // 4 * 4 + 8
    sino = np.full((3, my, sks), np.nan, np.float32)         # one matrix more than the angle list has
    sino[:2, :, :K] = rng.random((2, my, K)) - 0.3
    data = np.full((R + 1, my, CP), np.nan, np.float32)
    data[[1, 3]] = rng.random((2, my, CP)) - 0.3
    d_sino, d_data = torch.from_numpy(sino).cuda(), torch.from_numpy(data).cuda()
    rel = 3 * (max(K, CP) + 4) * 2.0 ** -23                  # as above
    for waves in (0, 32):
        out = torch.full((R, my, CP), 7.0, device="cuda")
        _lib.call("dfm_pfblk_forward", _lib.ptr(d_sino), sks, K, _lib.ptr(ptr), _lib.ptr(pos), _lib.ptr(val),
                  MODES[precision] + waves, _lib.ptr(inv), P, _lib.ptr(om), 2, my, CP, _lib.ptr(out), None, 1, 0, st)
        ref, mag = _product(sino[:2, :, :K], pf[[1, 3]], precision)
        assert np.all(np.abs(out.cpu().numpy()[[1, 3]] - ref) <= rel * mag)
        back = torch.full((2, my, sks), np.nan, device="cuda")
        _lib.call("dfm_pfblk_adjoint", _lib.ptr(d_data), _lib.ptr(ptr), _lib.ptr(pos), _lib.ptr(val),
                  MODES[precision] + waves, _lib.ptr(inv), P, _lib.ptr(om), 2, my, CP, K, _lib.ptr(back), sks, 1.0, st)
        back = back.cpu().numpy().astype(np.float64)
        ref, mag = _product(data[[1, 3]], pf[[1, 3]].transpose(0, 2, 1), precision)
        assert np.all(np.abs(back[:, :, :K] - ref) <= rel * mag) and np.all(back[:, :, K:] == 0.0)
