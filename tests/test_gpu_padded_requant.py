"""FP8 requant of rows that end inside a 128-element group, against the oracle
on zero-padded codes and scales: every byte, padding included."""
from types import SimpleNamespace

import numpy as np
import pytest
import torch

from helpers import bits_u8

pytestmark = pytest.mark.gpu
FP8 = torch.float8_e4m3fn


def _padded(q, s):
    kb = q.shape[1]
    pb = -(-kb // 64) * 64
    return (np.pad(q, ((0, 0), (0, pb - kb))), np.pad(s, ((0, 0), (0, pb // 16 - s.shape[1]))))


# K % 32 == 0: one to three blocks per row (fewer scale bytes than a dword);
# one, two, three blocks past a group; four groups (one tile) and more; row counts around the 8- and 16-row tiles, and enough
# of them for the 16-row tiles (2 * 256 tiles of 32 rows).
@pytest.mark.parametrize("M,K", [(2, 32), (7 * 2, 64), (16, 96), (8, 160), (9, 192 + 512), (18, 224), (130, 512 + 32),
                                 (17 * 2, 2880), (5600, 2880), (16386, 544)])
@pytest.mark.parametrize("spread", [3, 12, 255])
def test_padded_rows(oracle, dev, M, K, spread):
    import omo
    print("padded requant", M, K, spread, flush=True)
    r = np.random.default_rng(M + K + spread)
    q = r.integers(0, 256, (M, K // 2), dtype=np.uint8)
    s = r.integers(max(0, 128 - spread), min(255, 127 + spread) + 1, (M, K // 32)).astype(np.uint8)
    pq, ps = _padded(q, s)
    P = pq.shape[1] * 2
    if M * P // 2 % 128:
        pytest.skip("refused by the entry point: rows x padded bytes not a multiple of 128")
    out = torch.full((M, P), 0xAB, dtype=torch.uint8, device=dev).view(FP8)
    outs = torch.full((P // 128, M), float("nan"), dtype=torch.float32, device=dev)
    # a scale tensor that ends where its storage does, at any byte alignment
    flat = torch.empty(s.size + 1, dtype=torch.uint8, device=dev)
    sd = flat[1:].view(s.shape)
    sd.copy_(torch.from_numpy(s))
    omo.omo_Mxfp4ToFp8_padded(torch.from_numpy(q).to(dev), sd, out, outs)
    torch.cuda.synchronize()
    eo, es = oracle.mxfp4_to_fp8(pq, ps)
    np.testing.assert_array_equal(bits_u8(out).reshape(-1), np.asarray(eo).view(np.uint8).reshape(-1))
    np.testing.assert_array_equal(outs.cpu().numpy().view(np.uint32).reshape(-1),
                                  np.asarray(es).view(np.uint32).reshape(-1))


def test_wrapper_routes_agree(dev, monkeypatch):
    """The wrapper's in-kernel padding returns what its torch padding returns
    (values, shapes, strides), for the widths it takes; scales in other forms
    and refused shapes go the old way."""
    from omo_python_api import mxfp4_dequant as api
    g = torch.Generator().manual_seed(3)
    for M, half in ((256, 1440), (64, 48), (64, 16), (64, 56), (64, 96)):
        x = torch.randint(0, 256, (M, half), generator=g, dtype=torch.uint8).to(dev)
        s = torch.randint(120, 135, (M, -(-half // 16)), generator=g, dtype=torch.uint8).to(dev)
        forms = [s, torch.nn.functional.pad(s, (0, -s.shape[1] % 4))]
        if s.shape[1] % 4:  # strided scales are taken where padding makes them contiguous
            forms.append(s.t().contiguous().t())
        for sc in forms:
            got = api.omo_per_token_mxfp4ToFp8_wrapper(x, sc, [M // 2, M // 2])
            with monkeypatch.context() as mp:
                mp.setattr(api, "_pads_in_kernel", lambda *_: False)
                mp.setattr(api, "native", SimpleNamespace(requant=lambda *_: None))
                want = api.omo_per_token_mxfp4ToFp8_wrapper(x, sc, [M // 2, M // 2])
            for a, b in zip(got[0] + got[1], want[0] + want[1]):
                assert a.shape == b.shape and a.stride() == b.stride() and a.dtype == b.dtype
                assert torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8))
    assert api._pads_in_kernel(torch.zeros((2, 80), dtype=torch.uint8, device=dev),
                               torch.zeros((2, 5), dtype=torch.uint8, device=dev))
    with pytest.raises(RuntimeError):  # an odd row count of an odd number of groups
        api.omo_per_token_mxfp4ToFp8_wrapper(torch.zeros((3, 48), dtype=torch.uint8, device=dev),
                                             torch.zeros((3, 3), dtype=torch.uint8, device=dev), [3])
