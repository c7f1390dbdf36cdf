"""Per-split row->col FP8 with lengths passed by value: bit for bit against
the oracle at the edges of its tiles, orders and split counts, into outputs
pre-filled with a sentinel; the forms it refuses; and the wrapper's choice."""
import random

import numpy as np
import pytest
import torch

from helpers import bits_u8

pytestmark = pytest.mark.gpu
FP8 = torch.float8_e4m3fn


def _lens(n, total, seed):
    """n lengths (some 0) summing to total."""
    r = random.Random(seed)
    cuts = sorted(r.randint(0, total) for _ in range(n - 1))
    return [b - a for a, b in zip([0] + cuts, cuts + [total])]


def _payload(M, N, seed):
    r = np.random.default_rng(seed)
    return (r.integers(0, 256, (M, N // 2), dtype=np.uint8),
            r.integers(118, 136, (M, N // 32), dtype=np.uint8))


# One split and one row; zero lengths at both ends; 64 and 65 splits (one and
# two lengths per lane), 128 (the most); 16 and 17 column bands and 16 and 17
# splits (band walk and ranges), 17 and 64 of five row tiles each and of more
# on average (ranges and walk); widths with whole, partial and single-chunk last bands.
@pytest.mark.parametrize("lens,N", [([1], 32), ([0, 129, 0], 256), ([0, 0, 127, 128, 300, 0], 4352),
                                    (_lens(16, 900, 6), 4352), (_lens(17, 900, 7), 4352), (_lens(64, 900, 1), 4352),
                                    (_lens(65, 900, 2), 4352), (_lens(128, 1500, 3), 288),
                                    ([640] * 17, 4352), ([640] * 16 + [641], 4352), ([515, 640] * 32, 4384),
                                    ([0, 1280] * 32, 4384), ([0, 1281] * 31 + [0, 1537], 4384),
                                    (_lens(7, 2100, 4), 4096), (_lens(8, 4000, 5), 7040), ([512, 256], 4608)])
def test_value_splits_match_oracle(oracle, dev, lens, N):
    import omo
    print("value splits", len(lens), sum(lens), N, flush=True)
    M, srows = sum(lens), sum((m + 127) // 128 for m in lens)
    q, s = _payload(M, N, M + N)
    out_q = torch.full((M * N,), 0xAB, dtype=torch.uint8, device=dev).view(FP8)
    out_s = torch.full((srows, N), float("nan"), dtype=torch.float32, device=dev)
    omo.omo_Mxfp4RowToBf16ToFp8Col_splits(torch.from_numpy(q).to(dev), torch.from_numpy(s).to(dev), out_q, out_s, lens,
                                          1e-10)
    torch.cuda.synchronize()
    eo, es = oracle.row_to_fp8_col_msplit(q, s, lens)
    np.testing.assert_array_equal(bits_u8(out_q), eo)
    np.testing.assert_array_equal(out_s.cpu().numpy().view(np.uint32), es.view(np.uint32))


# The wrapper passes lengths by value up to 128 splits of 16 B aligned code
# rows and copies them to the device otherwise; both give the oracle's bytes.
@pytest.mark.parametrize("n,shift", [(128, 0), (129, 0), (5, 8)])
def test_wrapper_both_routes(oracle, dev, n, shift):
    from omo_python_api.mxfp4_dequant import omo_per_token_mxfp4RowToBf16ToFp8Col_msplit_wrapper as wrapper
    lens, N = _lens(n, 1000, n), 320
    q, s = _payload(1000, N, n)
    flat = torch.empty(q.size + 64, dtype=torch.uint8, device=dev)
    data = flat[shift:shift + q.size].view(q.shape)
    data.copy_(torch.from_numpy(q))
    ys, ss = wrapper(data, torch.from_numpy(s).to(dev), lens)
    torch.cuda.synchronize()
    eo, es = oracle.row_to_fp8_col_msplit(q, s, lens)
    assert [tuple(y.shape) for y in ys] == [(N, m) for m in lens]
    assert [tuple(x.shape) for x in ss] == [((m + 127) // 128, N) for m in lens]
    np.testing.assert_array_equal(np.concatenate([bits_u8(y).reshape(-1) for y in ys]), eo)
    np.testing.assert_array_equal(torch.cat(ss).cpu().numpy().view(np.uint32), es.view(np.uint32))


def test_refusals(dev):
    import omo
    N, M = 64, 256
    q = torch.zeros((M, N // 2), dtype=torch.uint8, device=dev)
    s = torch.full((M, N // 32), 127, dtype=torch.uint8, device=dev)
    out_q = torch.empty(M * N, dtype=torch.uint8, device=dev).view(FP8)
    out_s = torch.empty((200, N), dtype=torch.float32, device=dev)
    call = omo.omo_Mxfp4RowToBf16ToFp8Col_splits
    for bad in ([128, 127], [128, 129], [-1, 257]):
        with pytest.raises(RuntimeError):
            call(q, s, out_q, out_s, bad, 1e-10)
    with pytest.raises(RuntimeError, match="output_s"):
        call(q, s, out_q, out_s[:1], [128, 128], 1e-10)
    with pytest.raises(NotImplementedError):
        call(q, s, out_q, out_s, [2] * 127 + [1] * 2, 1e-10)
    with pytest.raises(NotImplementedError):
        call(q.view(-1)[8:8 + 128 * 32].view(128, 32), s[:128], out_q, out_s, [128], 1e-10)


def test_captured_replays(oracle, dev):
    """Lengths passed by value need no copy, so the whole wrapper captures;
    every replay reads the inputs of the moment."""
    from omo_python_api.mxfp4_dequant import omo_per_token_mxfp4RowToBf16ToFp8Col_msplit_wrapper as wrapper
    lens, N = [130, 0, 255, 1], 288
    q = torch.zeros((386, N // 2), dtype=torch.uint8, device=dev)
    s = torch.full((386, N // 32), 127, dtype=torch.uint8, device=dev)
    wrapper(q, s, lens)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ys, ss = wrapper(q, s, lens)
    for seed in range(3):
        hq, hs = _payload(386, N, seed)
        q.copy_(torch.from_numpy(hq))
        s.copy_(torch.from_numpy(hs))
        for t in ys + ss:
            t.view(torch.uint8).fill_(0xAB)
        graph.replay()
        torch.cuda.synchronize()
        eo, es = oracle.row_to_fp8_col_msplit(hq, hs, lens)
        np.testing.assert_array_equal(np.concatenate([bits_u8(y).reshape(-1) for y in ys]), eo)
        np.testing.assert_array_equal(torch.cat(ss).cpu().numpy().view(np.uint32), es.view(np.uint32))


# Tiles of 1 .. 128 rows: both sides of the 32- and 64-row forms, every count
# of bytes in a lane's last piece, outputs at every byte alignment; scale
# bytes of the fast path and of the restatement.
@pytest.mark.parametrize("lo,hi", [(118, 136), (0, 256)])
@pytest.mark.parametrize("N", [256, 352])
def test_rows_per_lane(oracle, dev, N, lo, hi):
    import omo
    for lens in (list(range(1, 40)) + [63, 64, 65, 66, 67], [128 + m for m in (1, 3, 31, 32, 33, 60, 64, 65, 97, 127)]):
        M, srows = sum(lens), sum((m + 127) // 128 for m in lens)
        r = np.random.default_rng(M + N)
        q = r.integers(0, 256, (M, N // 2), dtype=np.uint8)
        s = r.integers(lo, hi, (M, N // 32)).astype(np.uint8)
        out_q = torch.full((M * N,), 0xAB, dtype=torch.uint8, device=dev).view(FP8)
        out_s = torch.full((srows, N), float("nan"), dtype=torch.float32, device=dev)
        omo.omo_Mxfp4RowToBf16ToFp8Col_splits(torch.from_numpy(q).to(dev), torch.from_numpy(s).to(dev), out_q, out_s,
                                              lens, 1e-10)
        eo, es = oracle.row_to_fp8_col_msplit(q, s, lens)
        np.testing.assert_array_equal(bits_u8(out_q), eo)
        np.testing.assert_array_equal(out_s.cpu().numpy().view(np.uint32), es.view(np.uint32))
        for m in lens[::5]:  # the dense form of the same heights
            out_q, out_s = torch.empty((N, m), dtype=FP8, device=dev), torch.empty((-(-m // 128), N), device=dev)
            omo.omo_per_token_Mxfp4RowToBf16ToFp8Col(torch.from_numpy(q[:m]).to(dev), torch.from_numpy(s[:m]).to(dev),
                                                     out_q, out_s, 1e-10)
            eo, es = oracle.row_to_fp8_col(q[:m], s[:m])
            np.testing.assert_array_equal(bits_u8(out_q), eo)
            np.testing.assert_array_equal(out_s.cpu().numpy().view(np.uint32), es.view(np.uint32))
