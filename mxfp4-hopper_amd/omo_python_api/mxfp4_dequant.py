"""MXFP4 -> BF16 dequant and MXFP4 -> FP8 requant wrappers.

Mirrors code/kernel/api/mxfp4_dequant.py (padding, output allocation, slicing
and splitting) and adds the two wrappers the TE integration imports but the
reference does not ship:
  * omo_per_token_mxfp4RowToBf16ToFp8Col_wrapper (code/transformer_engine-2.8.diff:198, 259-272)
  * omo_per_token_mxfp4RowToBf16ToFp8Col_msplit_wrapper (code/transformer_engine-2.8.diff:70, 159-176)
Their contracts are reconstructed from those call sites and from the host
checks of the bound functions; eps = 1e-10 as in every shipped wrapper.

The wrappers that training calls try the native form of the same steps first
(csrc/binding/omo_native.cpp), which answers None where a call is not the
ordinary one.
"""
from typing import List

import torch
import torch.nn.functional as F

from omo import (
    DEQUANT_TYPES,
    omo_Mxfp4RowToBf16ToFp8Col_splits,
    omo_Mxfp4ToFp8_padded,
    omo_Mxfp4_dequant,
    omo_per_token_Mxfp4RowToBf16ToFp8Col,
    omo_per_token_Mxfp4RowToBf16ToFp8Col_msplit,
    omo_per_token_Mxfp4ToBf16ToFp8,
    omo_per_token_Mxfp4ToFp8,
    omo_per_token_Mxfp4ToFp8_col,
)
from omo._native import native

fp8_type_ = torch.float8_e4m3fn
uint8_type = torch.uint8
fp8_max = torch.finfo(fp8_type_).max
fp8_min = -fp8_max
mxfp4_max = 6.0
mxfp4_min = -mxfp4_max

FLOAT4_E2M1_MAX = 6.0
FLOAT8_E4M3_MAX = torch.finfo(torch.float8_e4m3fn).max


def pad_to_multiple(x, multiple=128):
    """Zero-pad the last dim to a multiple (mxfp4_dequant.py:15-29); returns
    (padded tensor, original last dim). No copy when already a multiple."""
    last_dim = x.shape[-1]
    pad_amount = (multiple - (last_dim % multiple)) % multiple
    x_padded = F.pad(x, (0, pad_amount)) if pad_amount > 0 else x
    return x_padded, last_dim


def unpad_from_multiple(x_padded, original_size):
    """mxfp4_dequant.py:31-33."""
    return x_padded[..., :original_size]


def omo_per_token_mxfp4ToBf16_dequant_wrapper(x: torch.Tensor, x_in_s: torch.Tensor, dtype):
    """codes [M, K/2] + scales [M, K/32] -> x_q.to(dtype) of shape [M, K]
    (mxfp4_dequant.py:39-74; called at code/transformer_engine-2.8.diff:392).
    fp16 and fp32 are written by the dequant itself; any other dtype is
    converted from bf16 in a second pass."""
    done = native.dequantize(x, x_in_s, dtype)
    if done is not None:
        return done
    group_size = 32
    assert x.shape[-1] % group_size == 0, "the last dimension of `x` cannot be divisible by `group_size`"
    assert x.is_contiguous(), "`x` is not contiguous"
    out_shape = (*x.shape[:-1], x.shape[-1] * 2)
    x_q = torch.empty(out_shape, device=x.device, dtype=dtype if dtype in DEQUANT_TYPES else torch.bfloat16)
    if x.shape[0] > 0:
        if x.dim() != 2:  # the reference's check of its scale output, shaped like x
            raise RuntimeError(f"Expected output_s.dim() == 2 ({x.dim()} vs. 2)")
        omo_Mxfp4_dequant(x, x_in_s, x_q)
    return x_q.to(dtype)


def omo_per_token_mxfp4ToBf16ToFp8_wrapper(x: torch.Tensor, x_in_s: torch.Tensor):
    """mxfp4_dequant.py:79-121: codes padded to 16 bytes, fp8 [M, 2Kp] sliced to
    [M, 2K], scales [2Kp/128, M] (TE layout)."""
    group_size = 128
    eps = 1e-10
    scale_ue8m0 = False
    x_padded, original_w = pad_to_multiple(x, multiple=16)
    assert x.is_contiguous(), "`x` is not contiguous"
    out_shape = (*x_padded.shape[:-1], x_padded.shape[-1] * 2)
    scale_shape = ((x_padded.shape[-1] * 2 // 128), *x_padded.shape[:-1])
    x_q = torch.empty(out_shape, device=x.device, dtype=fp8_type_)
    x_s = torch.empty(scale_shape, device=x.device, dtype=torch.float)
    if x.shape[0] > 0:
        omo_per_token_Mxfp4ToBf16ToFp8(x_padded, x_in_s, x_q, x_s, group_size, eps, mxfp4_min, mxfp4_max, scale_ue8m0)
    x_q = x_q[:, :original_w * 2]
    return x_q, x_s


def _pads_in_kernel(x: torch.Tensor, x_in_s: torch.Tensor) -> bool:
    """Whether the FP8 requant can read these rows unpadded: they end inside a
    128-element group, on a whole 32-element block, with one contiguous scale
    row of their own width each. Anything else is padded by torch first."""
    if x.dim() != 2 or x.shape[1] % 16 != 0:
        return False
    rows, half = x.shape
    return (tuple(x_in_s.shape) == (rows, half // 16) and x_in_s.is_contiguous() and x.dtype == x_in_s.dtype == uint8_type
            and x.is_cuda and x.device == x_in_s.device and x.data_ptr() % 8 == 0
            and rows * ((half + 63) // 64) % 2 == 0)  # what the kernel refuses is refused by the padded route


def omo_per_token_mxfp4ToFp8_wrapper(x: torch.Tensor, x_in_s: torch.Tensor, m_splits: List[int] = None):
    """mxfp4_dequant.py:122-187 (called at code/transformer_engine-2.8.diff:163):
    codes padded to 64 bytes and scales to 4 columns, fp8 [M, 2Kp] + fp32
    [2Kp/128, M], sliced, then split by m_splits along rows (fp8, dim 0) and
    columns (scales, dim 1). Widths K % 32 == 0 are padded inside the kernel."""
    done = native.requant(x, x_in_s, m_splits)
    if done is not None:
        return done
    group_size = 128
    eps = 1e-10
    scale_ue8m0 = False
    assert x.is_contiguous(), "`x` is not contiguous"
    original_w, original_w_scale = x.shape[-1], x_in_s.shape[-1]
    in_kernel = original_w % 64 != 0 and _pads_in_kernel(x, x_in_s)
    padded_w = (original_w + 63) // 64 * 64
    out_shape = (*x.shape[:-1], padded_w * 2)
    scale_shape = ((padded_w * 2 // 128), *x.shape[:-1])
    x_q = torch.empty(out_shape, device=x.device, dtype=fp8_type_)
    x_s = torch.empty(scale_shape, device=x.device, dtype=torch.float)
    if x.shape[0] > 0:
        if in_kernel:
            omo_Mxfp4ToFp8_padded(x, x_in_s, x_q, x_s)
        else:
            x_padded, _ = pad_to_multiple(x, multiple=64)
            x_in_s_pad, _ = pad_to_multiple(x_in_s, multiple=4)
            omo_per_token_Mxfp4ToFp8(x_padded, x_in_s_pad, x_q, x_s, group_size, eps, mxfp4_min, mxfp4_max,
                                     scale_ue8m0)
    x_q = x_q[:, :original_w * 2]
    # the reference slices the scale rows with the MX scale width
    # (mxfp4_dequant.py:172), which keeps every row
    x_s = x_s[:original_w_scale, :]
    x_q_split = torch.split(x_q, m_splits, dim=0)
    x_s_split = torch.split(x_s, m_splits, dim=1)
    return x_q_split, x_s_split


def omo_per_token_mxfp4ToFp8_col_wrapper(x: torch.Tensor, x_in_s: torch.Tensor):
    """mxfp4_dequant.py:189-237: codes padded to 16 bytes -> fp8 transposed
    [2Kp, M] (sliced on the last dim as the reference does) + fp32
    [M/128, 2Kp]."""
    group_size = 128
    eps = 1e-10
    scale_ue8m0 = False
    x_padded, original_w = pad_to_multiple(x, multiple=16)
    assert x.is_contiguous(), "`x` is not contiguous"
    out_shape = (x_padded.shape[-1] * 2, *x_padded.shape[:-1])
    scale_shape = ((x_padded.shape[0] // 128), x_padded.shape[-1] * 2)
    x_q = torch.empty(out_shape, device=x.device, dtype=fp8_type_)
    x_s = torch.empty(scale_shape, device=x.device, dtype=torch.float)
    if x.shape[0] > 0:
        omo_per_token_Mxfp4ToFp8_col(x_padded, x_in_s, x_q, x_s, group_size, eps, mxfp4_min, mxfp4_max, scale_ue8m0)
    x_q = x_q[..., :original_w * 2]
    return x_q, x_s


def omo_per_token_mxfp4RowToBf16ToFp8Col_wrapper(data: torch.Tensor, scale: torch.Tensor, eps: float = 1e-10):
    """Reconstructed wrapper of omo_per_token_Mxfp4RowToBf16ToFp8Col for TE's
    dense wgrad (code/transformer_engine-2.8.diff:259-272): codes [M, N/2] +
    scales [M, N/32] -> (fp8 columnwise data [N, M], fp32 columnwise
    scale_inv [ceil(M/128), N]) in TE's GEMM_READY layout."""
    done = native.row_to_col(data, scale, eps)
    if done is not None:
        return done
    assert data.dim() == 2 and data.is_contiguous(), "`data` must be a contiguous 2-D tensor"
    M, half = data.shape
    N = half * 2
    out_q = torch.empty((N, M), device=data.device, dtype=fp8_type_)
    out_s = torch.empty(((M + 127) // 128, N), device=data.device, dtype=torch.float)
    if M > 0 and N > 0:
        omo_per_token_Mxfp4RowToBf16ToFp8Col(data, scale.contiguous(), out_q, out_s, eps)
    return out_q, out_s


def split_metadata(m_splits: List[int], device) -> tuple:
    """int32 device tensors (lengths, row offsets, scale-row offsets) and the
    longest split, as the msplit kernel expects them
    (code/kernel/per_token_Mxfp4RowToBf16ToFp8Col_msplit.cu:74-80, 256)."""
    lens = [int(m) for m in m_splits]
    if any(m < 0 for m in lens):
        raise ValueError(f"m_splits must be non-negative, got {lens}")
    offs, soffs, o, so = [], [], 0, 0
    for m in lens:
        offs.append(o)
        soffs.append(so)
        o += m
        so += (m + 127) // 128
    meta = torch.tensor([lens, offs, soffs], dtype=torch.int32).to(device, non_blocking=False)
    return meta[0], meta[1], meta[2], (max(lens) if lens else 0), o, so


# Most splits that travel with the launch itself.
MAX_VALUE_SPLITS = 128


def omo_per_token_mxfp4RowToBf16ToFp8Col_msplit_wrapper(data: torch.Tensor, scale: torch.Tensor,
                                                        m_splits: List[int], eps: float = 1e-10):
    """Reconstructed wrapper of omo_per_token_Mxfp4RowToBf16ToFp8Col_msplit for
    TE's grouped wgrad (code/transformer_engine-2.8.diff:159-176): codes
    [sum(m), N/2] + scales -> (list of fp8 [N, m_i], list of fp32
    [ceil(m_i/128), N]), one per expert split, each a view of one buffer.

    Up to 128 splits of 16 B aligned code rows travel by value with the
    launch. More splits, rows the 256-column tiles do not take and tiles past
    one launch go through a device copy of the metadata, for which the host
    waits."""
    done = native.row_to_col_splits(data, scale, m_splits, eps)
    if done is not None:
        return done
    assert data.dim() == 2 and data.is_contiguous(), "`data` must be a contiguous 2-D tensor"
    total_m, half = data.shape
    N = half * 2
    lens = [int(m) for m in m_splits]
    if any(m < 0 for m in lens):
        raise ValueError(f"m_splits must be non-negative, got {lens}")
    rows, tiles = sum(lens), [(m + 127) // 128 for m in lens]
    if rows != total_m:
        raise ValueError(f"sum(m_splits)={rows} does not match data rows {total_m}")
    out_q = torch.empty(total_m * N, device=data.device, dtype=fp8_type_)
    out_s = torch.empty((sum(tiles), N), device=data.device, dtype=torch.float)
    if len(lens) > 0 and N > 0 and total_m > 0:
        scale = scale.contiguous()
        by_value = len(lens) <= MAX_VALUE_SPLITS and N % 32 == 0 and data.data_ptr() % 16 == 0 and total_m < 2**31
        if by_value:
            try:
                omo_Mxfp4RowToBf16ToFp8Col_splits(data, scale, out_q, out_s, lens, eps)
            except NotImplementedError:  # more tiles than a launch holds
                by_value = False
        if not by_value:
            meta, offs, soffs, max_len, _, _ = split_metadata(lens, data.device)
            omo_per_token_Mxfp4RowToBf16ToFp8Col_msplit(data, scale, out_q, out_s, meta, offs, soffs, max_len, eps)
    y_data, y_scale, o = [], [], 0
    for m in lens:
        y_data.append(out_q[o * N:(o + m) * N].view(N, m))
        o += m
    y_scale = list(torch.split(out_s, tiles, dim=0))
    return y_data, y_scale
