"""Dequant straight to fp16 and fp32: bit for bit the conversion of the bf16
dequant, which the oracle pins."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
TYPES = [torch.bfloat16, torch.float16, torch.float32]


def _bits(t):
    return t.contiguous().view(torch.int16 if t.element_size() == 2 else torch.int32)


def _want(oracle, dev, q, s, dtype):
    bf16 = torch.from_numpy(oracle.dequant_bf16(q.reshape(-1), s.reshape(-1)).view(np.int16)).view(torch.bfloat16)
    return bf16.to(dev).to(dtype)


@pytest.mark.parametrize("dtype", TYPES)
def test_every_code_and_scale(oracle, dev, dtype):
    """All 256 code bytes under all 256 scale bytes: zero, subnormal, overflow
    to inf, NaN of 0 * inf."""
    import omo
    q = np.tile(np.arange(256, dtype=np.uint8), (256, 1))
    s = np.repeat(np.arange(256, dtype=np.uint8)[:, None], 16, axis=1)
    out = torch.empty((256, 512), dtype=dtype, device=dev)
    omo.omo_Mxfp4_dequant(torch.from_numpy(q).to(dev), torch.from_numpy(np.ascontiguousarray(s)).to(dev), out)
    assert torch.equal(_bits(out).view(-1), _bits(_want(oracle, dev, q, s, dtype)))


# One unit past a workgroup's span, a tail of one block row, and sizes on both
# sides of one round of resident workgroups (8 x 256 of 1024 units).
@pytest.mark.parametrize("rows,K", [(2, 128), (1, 256), (33, 256), (4, 1024), (4096, 1024), (4097, 2048), (8200, 2048)])
@pytest.mark.parametrize("dtype", TYPES)
def test_sizes(oracle, dev, rows, K, dtype):
    from omo_python_api.ep_payload import join_payload, packed_mxfp4ToBf16
    from omo_python_api.mxfp4_dequant import omo_per_token_mxfp4ToBf16_dequant_wrapper as wrapper
    print("dequant", rows, K, dtype, flush=True)
    r = np.random.default_rng(rows + K)
    q = r.integers(0, 256, (rows, K // 2), dtype=np.uint8)
    s = r.integers(90, 160, (rows, K // 32), dtype=np.uint8)
    want = _bits(_want(oracle, dev, q, s, dtype))
    qd, sd = torch.from_numpy(q).to(dev), torch.from_numpy(s).to(dev)
    got = wrapper(qd, sd, dtype)
    assert got.dtype == dtype and got.shape == (rows, K)
    assert torch.equal(_bits(got).view(-1), want)
    assert torch.equal(_bits(packed_mxfp4ToBf16(join_payload(qd, sd), dtype)).view(-1), want)


def test_other_forms(dev):
    from omo_python_api.mxfp4_dequant import omo_per_token_mxfp4ToBf16_dequant_wrapper as wrapper
    q = torch.randint(0, 256, (4, 64), dtype=torch.uint8, device=dev)
    s = torch.full((4, 4), 130, dtype=torch.uint8, device=dev)
    assert torch.equal(wrapper(q, s, torch.float64), wrapper(q, s, torch.bfloat16).double())
    with pytest.raises(RuntimeError, match="dim"):
        wrapper(q.view(2, 2, 64), s.view(2, 2, 4), torch.float32)
