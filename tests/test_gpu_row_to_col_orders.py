"""Dense row->col FP8 on ragged row counts in each of its tile orders (bands
fastest, rows fastest, band walk), on both sides of the lines between them,
into outputs pre-filled with a sentinel: every byte against the oracle."""
import numpy as np
import pytest
import torch

from helpers import bits_u8

pytestmark = pytest.mark.gpu
FP8 = torch.float8_e4m3fn


# On 256 CUs: up to 160 tiles bands fastest, up to 1280 rows fastest, more
# the band walk. One band and many; whole and partial last bands; row
# counts one past and one short of whole tiles, and 16 B aligned columns that
# are not whole lines.
@pytest.mark.parametrize("M,N", [(128 * 159 + 1, 256), (128 * 160 + 1, 256), (129, 128 * 257), (1000, 2880),
                                 (128 * 6 - 1, 7168), (128 * 96 + 16, 4000), (128 * 1279 + 3, 256),
                                 (128 * 1280 + 3, 256), (128 * 768 - 5, 288), (128 * 96 + 48, 4160),
                                 # past 1280 tiles: one tile of at most 64 rows bands fastest, of more and up to
                                 # eight row tiles rows fastest; five bands past 3584 tiles bands fastest, not past:
                                 # the walk; up to 16 bands past 3072 tiles the walk without the LDS reserve
                                 (33, 256 * 1281), (64, 256 * 1281 + 32), (65, 256 * 1281), (1001, 256 * 161 + 96),
                                 (1025, 256 * 143), (128 * 716 + 1, 1280), (128 * 717 + 1, 1280), (128 * 512 + 1, 1536),
                                 (128 * 193 + 77, 4096)])
def test_ragged_orders(oracle, dev, M, N):
    import omo
    print("ragged order", M, N, flush=True)
    r = np.random.default_rng(M + N)
    q = r.integers(0, 256, (M, N // 2), dtype=np.uint8)
    s = r.integers(118, 136, (M, N // 32), dtype=np.uint8)
    out = torch.full((N, M), 0xAB, dtype=torch.uint8, device=dev).view(FP8)
    outs = torch.full((-(-M // 128), N), float("nan"), dtype=torch.float32, device=dev)
    omo.omo_per_token_Mxfp4RowToBf16ToFp8Col(torch.from_numpy(q).to(dev), torch.from_numpy(s).to(dev), out, outs, 1e-10)
    torch.cuda.synchronize()
    eo, es = oracle.row_to_fp8_col(q, s)
    np.testing.assert_array_equal(bits_u8(out), eo)
    np.testing.assert_array_equal(outs.cpu().numpy().view(np.uint32), es.view(np.uint32))
