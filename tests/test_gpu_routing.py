"""The row map of a routing map by the HIP kernels against the torch
composition of the same map on the CPU: whole numbers, so every value."""
import numpy as np
import pytest
import torch

from helpers import bits_u8

pytestmark = pytest.mark.gpu


def _map(T, E, p, seed):
    return torch.rand((T, E), generator=torch.Generator().manual_seed(seed)) < p


# One token, one expert; experts that are not a multiple of the four of a
# workgroup; token counts around a wave (64), a workgroup step (256) and
# several steps per chunk (more than 64 or, with many experts, 8 chunks);
# nothing routed and everything routed.
@pytest.mark.parametrize("T,E,p", [(1, 1, 1.0), (1, 1, 0.0), (63, 3, 0.5), (64, 4, 0.3), (65, 5, 1.0), (256, 64, 0.125),
                                   (257, 6, 0.4), (4096, 64, 0.125), (16640, 8, 0.2), (40000, 2, 0.5),
                                   (5000, 520, 0.02)])
@pytest.mark.parametrize("pad", [None, 0, 7, 3000])
def test_row_map(dev, T, E, p, pad):
    from omo_python_api.permutation import make_row_id_map
    print("row map", T, E, p, pad, flush=True)
    rm = _map(T, E, p, T + E)
    num_out = None if pad is None else int(rm.sum()) + pad
    src, m_splits, dest = make_row_id_map(rm.to(dev), num_out)
    es, em, ed = make_row_id_map(rm, num_out)
    assert m_splits == em and all(isinstance(m, int) for m in m_splits)
    assert src.dtype == es.dtype and dest.dtype == ed.dtype and src.is_contiguous()
    assert torch.equal(src.cpu(), es) and torch.equal(dest.cpu(), ed)
    assert src.untyped_storage().nbytes() == 4 * src.numel()


# Both sides of the maps that the torch composition does faster: one and two
# experts of very many tokens, and very many experts (3 chunks of tokens).
@pytest.mark.parametrize("T,E,p,takes", [(2**22 - 1, 1, 0.5, True), (2**22, 1, 0.5, False), (2**23 - 1, 2, 0.3, True),
                                         (2**23, 2, 0.3, False), (2**22, 3, 0.3, True), (700, 43690, 2e-4, True),
                                         (700, 43691, 2e-4, False)])
def test_row_map_routes(dev, T, E, p, takes):
    from omo._native import native
    from omo_python_api.permutation import make_row_id_map
    print("row map route", T, E, flush=True)
    rm = _map(T, E, p, T + E)
    rmd = rm.to(dev)
    assert (native.make_row_map(rmd, None) is not None) == takes
    src, m_splits, dest = make_row_id_map(rmd)
    es, em, ed = make_row_id_map(rm)
    assert m_splits == em and torch.equal(src.cpu(), es) and torch.equal(dest.cpu(), ed)


def test_row_map_forms(dev):
    """Strided and misaligned maps, 0/1 maps of other types, too few rows."""
    from omo_python_api.permutation import make_row_id_map
    rm = _map(300, 12, 0.3, 1)
    es, em, ed = make_row_id_map(rm)
    wide = torch.zeros((300, 20), dtype=torch.bool, device=dev)
    wide[:, 3:15] = rm.to(dev)
    flat = torch.zeros(300 * 12 + 1, dtype=torch.bool, device=dev)
    flat[1:] = rm.to(dev).view(-1)
    forms = [wide[:, 3:15], flat[1:].view(300, 12), rm.to(dev).t().contiguous().t(), rm.to(dev).int(), rm.to(dev).float()]
    for f in forms:
        src, m_splits, dest = make_row_id_map(f)
        assert m_splits == em and torch.equal(src.cpu(), es) and torch.equal(dest.cpu(), ed)
    with pytest.raises(ValueError, match="smaller"):
        make_row_id_map(rm.to(dev), int(rm.sum()) - 1)
    for T, E in ((0, 4), (4, 0)):
        src, m_splits, dest = make_row_id_map(torch.zeros((T, E), dtype=torch.bool, device=dev), 3)
        assert src.tolist() == [-1] * 3 and m_splits == [0] * E and dest.shape == (T, E)


# The row order that the fused requant copies out of its scratch (no row count
# given): the 8-row tile and the 32-row one (from 512 tiles), with one column
# of workgroups and with three (only the first copies), the last tile whole and
# of 2, 7, 12 and 13 rows; on the current stream and on another.
@pytest.mark.parametrize("T,H,E,k", [(301, 128, 12, 3), (4099, 128, 16, 4), (4096, 128, 8, 4), (2742, 1152, 8, 3),
                                     (2735, 1280, 64, 3)])
@pytest.mark.parametrize("side", [False, True])
def test_copied_row_order(oracle, dev, T, H, E, k, side):
    from omo._native import native
    from omo_python_api.permutation import mxfp4_permute_to_fp8
    print("copied row order", T, H, E, k, side, flush=True)
    g = torch.Generator().manual_seed(T + H)
    rm = torch.zeros((T, E), dtype=torch.bool).scatter_(1, torch.rand((T, E), generator=g).topk(k, dim=1).indices, True)
    q = torch.randint(0, 256, (T, H // 2), generator=g, dtype=torch.uint8)
    s = torch.randint(118, 136, (T, H // 32), generator=g, dtype=torch.uint8)
    e_idx, t_idx = np.nonzero(rm.numpy().T)
    eo, es = oracle.mxfp4_to_fp8(q.numpy()[t_idx], s.numpy()[t_idx])
    qd, sd, rmd = q.to(dev), s.to(dev), rm.to(dev)
    torch.cuda.synchronize()
    with torch.cuda.stream(torch.cuda.Stream() if side else torch.cuda.current_stream()):
        assert native.permute_to_fp8(qd, sd, rmd, None) is not None
        for _ in range(2):  # the second call finds the first one's scratch in the allocator
            f8, f8s, src, m_splits = mxfp4_permute_to_fp8(qd, sd, rmd, split=False)
        torch.cuda.current_stream().synchronize()
    assert m_splits == np.bincount(e_idx, minlength=E).tolist()
    assert src.dtype == torch.int32 and src.untyped_storage().nbytes() == 4 * src.numel()
    np.testing.assert_array_equal(src.cpu().numpy(), t_idx)
    np.testing.assert_array_equal(bits_u8(f8), eo)
    np.testing.assert_array_equal(f8s.cpu().numpy().view(np.uint32), es.view(np.uint32))
