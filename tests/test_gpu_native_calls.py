"""The native form of the wrappers' calls against their Python form (native
answering None): the same values, types, shapes and strides where it takes a
call, and the same answer or error where it does not."""
from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu


class _Sub(torch.Tensor):
    pass


def _apis():
    from omo_python_api import ep_payload, mxfp4, mxfp4_dequant, permutation
    return mxfp4, mxfp4_dequant, ep_payload, permutation


def _tree(v):
    if isinstance(v, torch.Tensor):
        return ("tensor", type(v), v.dtype, tuple(v.shape), v.stride(), v.storage_offset(), v.device, v.requires_grad,
                v._is_view(), v.contiguous().view(torch.uint8).flatten().tolist() if v.numel() else [])
    if isinstance(v, (list, tuple)):
        return (type(v), [_tree(x) for x in v])
    return v


def _outcome(call):
    try:
        return _tree(call())
    except Exception as e:  # noqa: BLE001 (the two forms are compared by what they raise)
        return type(e)


def _both(call, monkeypatch):
    """Outcomes of a call in its native and in its Python form."""
    got = _outcome(call)
    with monkeypatch.context() as mp:
        for api in _apis():
            mp.setattr(api, "native", SimpleNamespace(**{n: (lambda *_: None) for n in dir(api.native) if n[0] != "_"}))
        return got, _outcome(call)


def _bf16(dev, *shape):
    return torch.randn(shape, generator=torch.Generator().manual_seed(7)).to(torch.bfloat16).to(dev)


def _u8(dev, lo, hi, *shape):
    return torch.randint(lo, hi, shape, generator=torch.Generator().manual_seed(9), dtype=torch.uint8).to(dev)


def _calls(dev):
    """name -> call: ordinary calls, odd ones and refused ones."""
    mx, de, ep, pe = _apis()
    x = _bf16(dev, 64, 256)
    forms = {"plain": x, "parameter": torch.nn.Parameter(x.clone()), "strided": _bf16(dev, 256, 64).t(),
             "row view": _bf16(dev, 70, 256)[3:67], "misaligned": _bf16(dev, 64 * 256 + 1)[1:].view(64, 256),
             "3-D": x.view(2, 32, 256), "1-D": x.view(-1), "no rows": x[:0], "no columns": x[:, :0].contiguous(),
             "width 33": _bf16(dev, 64, 33), "rows 33": _bf16(dev, 33, 256), "float": x.float(), "cpu": x.cpu(),
             "subclass": x.as_subclass(_Sub), "not a tensor": [1.0]}
    calls = {}
    for n, t in forms.items():
        calls["quantize " + n] = lambda t=t: mx.omo_per_token_group_quant_mxfp4(t)
        calls["dual " + n] = lambda t=t: mx.omo_per_token_group_quant_mxfp4_dual(t)
        calls["grouped " + n] = lambda t=t: mx.omo_per_token_group_quant_mxfp4_dual_grouped([x, t])
        calls["packed " + n] = lambda t=t: ep.fp4_quantize_packed(t)
    for n, eps in (("int", 1), ("nan", float("nan")), ("inf", float("inf")), ("huge", 1e300), ("large", 2.0),
                   ("negative", -1.0), ("text", "1")):
        calls["dual eps " + n] = lambda e=eps: mx.omo_per_token_group_quant_mxfp4_dual(x, e)
        calls["packed eps " + n] = lambda e=eps: ep.fp4_quantize_packed(x, e)
    calls["grouped tuple"] = lambda: mx.omo_per_token_group_quant_mxfp4_dual_grouped((x, x[:32]))
    calls["grouped none"] = lambda: mx.omo_per_token_group_quant_mxfp4_dual_grouped([])
    calls["grouped generator"] = lambda: mx.omo_per_token_group_quant_mxfp4_dual_grouped(t for t in (x,))

    q, s = _u8(dev, 0, 256, 48, 128), _u8(dev, 120, 131, 48, 8)
    codes = {"plain": (q, s), "padded width": (_u8(dev, 0, 256, 48, 80), _u8(dev, 120, 131, 48, 5)),
             "odd rows": (_u8(dev, 0, 256, 47, 64), _u8(dev, 120, 131, 47, 4)), "width 24": (q[:, :24].contiguous(), s[:, :2]),
             "strided codes": (q.t().contiguous().t(), s), "strided scales": (q, s.t().contiguous().t()),
             "few scales": (q, s[:, :7].contiguous()), "many scales": (q, _u8(dev, 120, 131, 128, 8)),
             "flat scales": (q, s.view(-1)), "int8 codes": (q.view(torch.int8), s), "float scales": (q, s.float()),
             "cpu scales": (q, s.cpu()), "cpu": (q.cpu(), s.cpu()), "3-D": (q.view(2, 24, 128), s.view(2, 24, 8)),
             "no rows": (q[:0], s[:0]), "misaligned": (_u8(dev, 0, 256, 48 * 128 + 4)[4:].view(48, 128), s),
             "shifted scales": (q, _u8(dev, 120, 131, 48 * 8 + 1)[1:].view(48, 8)),
             "subclass": (q.as_subclass(_Sub), s)}
    for n, (c, k) in codes.items():
        m = c.shape[0]
        splits = [m // 3, 0, m - m // 3]
        for dt in (torch.bfloat16, torch.float16, torch.float32, torch.float64):
            calls[f"dequant {n} {dt}"] = lambda c=c, k=k, dt=dt: de.omo_per_token_mxfp4ToBf16_dequant_wrapper(c, k, dt)
        calls["requant " + n] = lambda c=c, k=k, sp=splits: de.omo_per_token_mxfp4ToFp8_wrapper(c, k, sp)
        calls["row_to_col " + n] = lambda c=c, k=k: de.omo_per_token_mxfp4RowToBf16ToFp8Col_wrapper(c, k)
        calls["splits " + n] = lambda c=c, k=k, sp=splits: de.omo_per_token_mxfp4RowToBf16ToFp8Col_msplit_wrapper(c, k, sp)
        calls["payload " + n] = lambda c=c, k=k, sp=splits: ep.packed_mxfp4ToFp8(torch.cat((c, k), dim=-1), sp)
    for n, sp in (("tuple", (16, 32)), ("short", [16, 31]), ("long", [16, 33]), ("negative", [50, -2]), ("floats", [16.0, 32.0]),
                  ("bools", [True, 47]), ("int", 16), ("none", None), ("tensor", torch.tensor([16, 32])), ("one", [48]),
                  ("ones", [1] * 48), ("empty", []), ("129", [48] + [0] * 128)):
        calls["requant splits " + n] = lambda sp=sp: de.omo_per_token_mxfp4ToFp8_wrapper(q, s, sp)
        calls["row_to_col splits " + n] = lambda sp=sp: de.omo_per_token_mxfp4RowToBf16ToFp8Col_msplit_wrapper(q, s, sp)
        calls["payload splits " + n] = lambda sp=sp: ep.packed_mxfp4ToFp8(torch.cat((q, s), dim=-1), sp)
    for eps in (1, float("nan"), float("inf"), 500.0):
        calls[f"row_to_col eps {eps}"] = lambda e=eps: de.omo_per_token_mxfp4RowToBf16ToFp8Col_wrapper(q, s, e)
        calls[f"splits eps {eps}"] = lambda e=eps: de.omo_per_token_mxfp4RowToBf16ToFp8Col_msplit_wrapper(q, s, [48], e)

    payload = torch.cat((q, s), dim=-1)
    vq, vs = pe.payload_views(payload)
    rm = (torch.rand((48, 6), generator=torch.Generator().manual_seed(3)) < 0.4).to(dev)
    n = int(rm.sum())
    for name, m in (("bool", rm), ("int", rm.int()), ("strided", rm.t().contiguous().t()), ("cpu", rm.cpu()), ("none", rm & False),
                    ("fewer tokens", rm[:40]), ("subclass", rm.as_subclass(_Sub)), ("1-D", rm.view(-1)),
                    ("no experts", rm[:, :0])):
        for k in (None, n + 5, n, 3, 0, -1):
            calls[f"row map {name} {k}"] = lambda m=m, k=k: pe.make_row_id_map(m, k)
            calls[f"permute {name} {k}"] = lambda m=m, k=k: pe.mxfp4_permute_to_fp8(q, s, m, k)
    calls["permute views"] = lambda: pe.mxfp4_permute_to_fp8(vq, vs, rm)
    calls["permute unsplit"] = lambda: pe.mxfp4_permute_to_fp8(q, s, rm, split=False)
    calls["permute short scales"] = lambda: pe.mxfp4_permute_to_fp8(q, s[:, :7], rm)
    calls["permute width"] = lambda: pe.mxfp4_permute_to_fp8(q[:, :80], s[:, :5], rm)
    calls["permute fewer codes"] = lambda: pe.mxfp4_permute_to_fp8(q[:20], s[:20], rm)
    return calls


def test_native_and_python_forms_agree(dev, monkeypatch):
    bad = []
    for name, call in _calls(dev).items():
        got, want = _both(call, monkeypatch)
        if got != want:
            bad.append(name)
    assert not bad, bad


def test_ordinary_calls_are_native(dev):
    from omo._native import native
    x, q, s = _bf16(dev, 64, 256), _u8(dev, 0, 256, 48, 128), _u8(dev, 120, 131, 48, 8)
    rm = torch.ones((48, 4), dtype=torch.bool, device=dev)
    for r in (native.quantize(x), native.quantize_dual(x, 1e-10), native.quantize_dual_grouped([x], 1e-10),
              native.dequantize(q, s, torch.float32), native.requant(q, s, [48]), native.row_to_col(q, s, 1e-10),
              native.row_to_col_splits(q, s, [20, 28], 1e-10), native.quantize_packed(x, 1e-10),
              native.requant_packed(torch.cat((q, s), 1), None), native.make_row_map(rm, None),
              native.permute_to_fp8(q, s, rm, None)):
        assert r is not None


def test_modes_and_transforms_take_the_python_form(dev):
    """A torch-function or dispatch mode, fake tensors and vmap see the calls
    they saw before."""
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    from omo._native import native
    from omo_python_api.mxfp4 import omo_per_token_group_quant_mxfp4 as quantize
    x = _bf16(dev, 64, 256)

    class Functions(TorchFunctionMode):
        seen = 0

        def __torch_function__(self, func, types, args=(), kwargs=None):
            Functions.seen += func is torch.empty
            return func(*args, **(kwargs or {}))

    class Dispatch(TorchDispatchMode):
        seen = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            Dispatch.seen += func.overloadpacket is torch.ops.aten.empty
            return func(*args, **(kwargs or {}))

    for mode in (Functions, Dispatch):
        with mode():
            assert native.quantize(x) is None
            quantize(x)
        assert mode.seen == 2
    assert native.quantize(x) is not None

    def inside(t):
        assert native.quantize(t) is None and native.quantize(x) is None
        return t

    torch.vmap(inside)(x.view(2, 32, 256))


def test_side_stream_and_threads(dev):
    """Calls on a side stream and from two threads return each thread's values."""
    import threading

    from omo_python_api.mxfp4 import omo_per_token_group_quant_mxfp4 as quantize
    from omo_python_api.permutation import make_row_id_map
    xs = [_bf16(dev, 96, 512) * (i + 1) for i in range(2)]
    maps = [(torch.rand((500, 9), generator=torch.Generator().manual_seed(i)) < 0.3).to(dev) for i in range(2)]
    want = [([t.clone() for t in quantize(x)], make_row_id_map(m.cpu())) for x, m in zip(xs, maps)]
    torch.cuda.synchronize()
    wrong = []

    def work(i):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for _ in range(20):
                got, rows = quantize(xs[i]), make_row_id_map(maps[i])
                stream.synchronize()
                if not (all(torch.equal(a, b) for a, b in zip(got, want[i][0])) and rows[1] == want[i][1][1]
                        and torch.equal(rows[0].cpu(), want[i][1][0])):
                    wrong.append(i)

    ts = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not wrong


@pytest.mark.parametrize("num_out", [None, 1 << 24])
def test_refused_row_order_leaves_pinned_memory_alone(dev, num_out):
    """A permute whose row order (64 MB here) does not fit the device raises
    out of memory; no launch of it writes host memory afterwards, which the
    next pinned tensor of the counts' size would show, and the next call is
    right."""
    from omo_python_api.permutation import mxfp4_permute_to_fp8
    T, E, chunks = 16384, 1024, 8
    print("refused row order", num_out, flush=True)
    q, s = _u8(dev, 0, 256, T, 64), _u8(dev, 120, 131, T, 4)
    rm = torch.zeros((T, E), dtype=torch.bool, device=dev)
    rm[::7, 5] = True
    want = mxfp4_permute_to_fp8(q, s, rm, split=False)
    want = [t.cpu() for t in want[:3]] + [want[3]]
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(dev).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (40 << 20)) / total)
    try:
        torch.cuda._sleep(50 * 2_400_000)  # what the call enqueues starts after the host is done below
        with pytest.raises(torch.cuda.OutOfMemoryError):
            mxfp4_permute_to_fp8(q, s, rm, num_out, split=False)
        next_pinned = torch.empty((E * chunks,), dtype=torch.int32, pin_memory=True).fill_(-7)
        torch.cuda.synchronize()
        assert (next_pinned == -7).all()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    got = mxfp4_permute_to_fp8(q, s, rm, split=False)
    for a, b in zip(got[:3], want[:3]):
        assert torch.equal(a.cpu().view(torch.uint8), b.view(torch.uint8))
    assert got[3] == want[3]


@pytest.mark.parametrize("name", ["quantize", "dual", "grouped", "dequant", "requant", "row_to_col", "splits", "packed",
                                  "requant packed", "row map", "permute"])
def test_other_threads_run_while_a_call_allocates(dev, name):
    """A call whose outputs fit only once cached memory is freed waits for the
    device inside its allocation; other Python threads run meanwhile."""
    import threading
    import time
    mx, de, ep, pe = _apis()
    print("threads while", name, flush=True)
    M, K = 8192, 8192
    x = torch.zeros((M, K), dtype=torch.bfloat16, device=dev)
    q, s = torch.zeros((M, K // 2), dtype=torch.uint8, device=dev), torch.full((M, K // 32), 127, dtype=torch.uint8, device=dev)
    payload, rm = torch.cat((q, s), 1), torch.zeros((M, 1024), dtype=torch.bool, device=dev)
    rm[:, 3] = True
    call = {"quantize": lambda: mx.omo_per_token_group_quant_mxfp4(x),
            "dual": lambda: mx.omo_per_token_group_quant_mxfp4_dual(x),
            "grouped": lambda: mx.omo_per_token_group_quant_mxfp4_dual_grouped([x]),
            "dequant": lambda: de.omo_per_token_mxfp4ToBf16_dequant_wrapper(q, s, torch.float32),
            "requant": lambda: de.omo_per_token_mxfp4ToFp8_wrapper(q, s, [M]),
            "row_to_col": lambda: de.omo_per_token_mxfp4RowToBf16ToFp8Col_wrapper(q, s),
            "splits": lambda: de.omo_per_token_mxfp4RowToBf16ToFp8Col_msplit_wrapper(q, s, [M]),
            "packed": lambda: ep.fp4_quantize_packed(x),
            "requant packed": lambda: ep.packed_mxfp4ToFp8(payload, [M]),
            "row map": lambda: pe.make_row_id_map(rm),
            "permute": lambda: pe.mxfp4_permute_to_fp8(q[:, :64], s[:, :4], rm)}[name]
    call()  # its kernels are loaded
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    # 480 MB in free pieces smaller than the outputs, none beside another
    pieces = [torch.empty(12 << 20, dtype=torch.uint8, device=dev) for _ in range(80)]
    total = torch.cuda.get_device_properties(dev).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (1 << 20)) / total)
    ticks, stop = [], threading.Event()

    def tick():
        while not stop.wait(0.001):
            ticks.append(time.perf_counter())

    thread = threading.Thread(target=tick)
    try:
        del pieces[::2]
        torch.cuda._sleep(200 * 2_400_000)
        thread.start()
        t0 = time.perf_counter()
        call()
        t1 = time.perf_counter()
    finally:
        stop.set()
        thread.join()
        torch.cuda.set_per_process_memory_fraction(1.0)
        torch.cuda.synchronize()
    assert t1 - t0 > 0.05, "the allocation did not wait"
    assert sum(t0 < t < t1 for t in ticks) > 20 * (t1 - t0) / 0.1, (t1 - t0, len(ticks))


@pytest.mark.parametrize("fused", [False, True])
def test_row_map_refuses_a_capturing_stream(dev, fused):
    """The row map needs the host, so a capture refuses it before anything of
    it is recorded; the capture goes on, and its replays touch no pinned memory."""
    from omo_python_api.permutation import make_row_id_map, mxfp4_permute_to_fp8
    print("row map under capture", fused, flush=True)
    T, E = 4096, 16
    q, s = _u8(dev, 0, 256, T, 64), _u8(dev, 120, 131, T, 4)
    rm = torch.zeros((T, E), dtype=torch.bool, device=dev)
    rm[::3, 2] = True
    call = (lambda: mxfp4_permute_to_fp8(q, s, rm)) if fused else (lambda: make_row_id_map(rm))
    call()
    x = torch.zeros(4, device=dev)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        x += 1
        with pytest.raises(RuntimeError, match="captured"):
            call()
        x += 1
    pinned = torch.empty((E * 16,), dtype=torch.int32, pin_memory=True).fill_(-7)  # of the counts' size
    for _ in range(2):
        graph.replay()
    torch.cuda.synchronize()
    assert x.tolist() == [4.0] * 4 and (pinned == -7).all()
    call()
