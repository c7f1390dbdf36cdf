"""Dual-layout quantize on tensors of whole 64 x 256 tiles and just short of
them, with scale buffers at odd addresses and rows of an odd number of scale
bytes: every byte, and none around, against the rowwise oracle of x and of its
transpose, alone and grouped."""
import numpy as np
import pytest
import torch

from helpers import bits_u16, bits_u8

pytestmark = pytest.mark.gpu


def _outs(dev, M, K, row_shift, col_shift):
    def buf(rows, cols, shift):
        flat = torch.full((rows * cols + 16,), 0xAB, dtype=torch.uint8, device=dev)
        return flat[shift:shift + rows * cols].view(rows, cols)
    return (buf(M, K // 2, 0), buf(M, K // 32, row_shift), buf(K, M // 2, 0), buf(K, M // 32, col_shift))


def _check(oracle, x, outs):
    M, K = x.shape
    for bits, q, s in ((bits_u16(x), outs[0], outs[1]), (bits_u16(x.t()), outs[2], outs[3])):
        eq, es = oracle.quant_mxfp4(np.ascontiguousarray(bits).reshape(-1))
        np.testing.assert_array_equal(bits_u8(q).reshape(-1), np.asarray(eq).reshape(-1))
        np.testing.assert_array_equal(bits_u8(s).reshape(-1), np.asarray(es).reshape(-1))


# one tile; two of each; an inf block (the restated path); one tile short of
# whole in each direction; 9 and 15 scale bytes per row, 3 and 5 per column
@pytest.mark.parametrize("M,K", [(64, 256), (128, 512), (96, 256), (64, 288), (160, 480)])
@pytest.mark.parametrize("row_shift,col_shift", [(0, 0), (4, 0), (0, 1), (3, 5)])
def test_whole_tiles(oracle, dev, M, K, row_shift, col_shift):
    import omo
    print("dual whole tiles", M, K, row_shift, col_shift, flush=True)
    x = torch.randn((M, K), generator=torch.Generator().manual_seed(M + K)).to(torch.bfloat16)
    x[3, 40], x[33, 7] = float("inf"), 0.0
    outs = _outs(dev, M, K, row_shift, col_shift)
    grouped = [_outs(dev, M, K, row_shift, col_shift), _outs(dev, M, K, 0, 0)]
    xd = x.to(dev)
    omo.omo_quant_mxfp4_dual(xd, *outs)
    omo.omo_quant_mxfp4_dual_grouped([xd, xd], grouped)
    torch.cuda.synchronize()
    for o in [outs] + grouped:
        _check(oracle, x, o)
        for buf in o:  # nothing before or after the buffer was written
            whole = torch.as_strided(buf, (buf.untyped_storage().nbytes(),), (1,), 0)
            at = buf.storage_offset()
            assert (whole[:at] == 0xAB).all() and (whole[at + buf.numel():] == 0xAB).all()


# The orders of the tiles: ranges (few tiles), band groups in units of four
# tiles with a last row of units of one to four (6 tiles per CU: 1536 tiles),
# tensors of only such a row, and grouped items of at most and of more than 64
# bands side by side.
@pytest.mark.parametrize("M,K", [(64 * 23, 256 * 67), (64 * 24, 256 * 64), (64 * 25 + 32, 256 * 62 + 32), (64 * 1538, 256),
                                 (32, 256 * 1537), (64 * 2, 256 * 771), (64 * 3 - 32, 256 * 512 + 64), (64 * 4, 256 * 385),
                                 (64 * 5, 256 * 311), (64 * 7, 256 * 220)])
def test_orders(oracle, dev, M, K):
    import omo
    print("dual order", M, K, flush=True)
    x = torch.randn((M, K), generator=torch.Generator().manual_seed(K)).to(torch.bfloat16)
    xd = x.to(dev)
    outs = _outs(dev, M, K, 0, 0)
    omo.omo_quant_mxfp4_dual(xd, *outs)
    R = min(M, 160)
    small = xd[:R, :].contiguous()
    grouped = [_outs(dev, R, K, 0, 0), _outs(dev, M, K, 0, 0), _outs(dev, R, K, 0, 0)]
    omo.omo_quant_mxfp4_dual_grouped([small, xd, small], grouped)
    torch.cuda.synchronize()
    _check(oracle, x, outs)
    for a, b in zip(outs, grouped[1]):
        assert torch.equal(a, b)
    for o in (grouped[0], grouped[2]):
        _check(oracle, x[:R], o)
