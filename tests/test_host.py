"""The native calls behind the layer-level entry points (sglang_amd._host).

They must decline - return None before launching anything - whatever they do not take as it is, so that the dispatcher path
decides; and where they do take a call, its result is that of the dispatcher path, bit for bit.
"""
import sys
import threading
import time
import types

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.overrides import TorchFunctionMode

from sglang_amd import _host, fp8_kernel, fp8_utils, fused_moe, sgl_kernel

BLOCK = [128, 128]


def test_declines_what_it_does_not_take():
    x, w, s = torch.zeros((4, 256), dtype=torch.bfloat16), torch.zeros((128, 256), dtype=torch.float8_e4m3fn), torch.ones((1, 2))
    assert _host.block_linear(x, w, BLOCK, s, None) is None  # host memory
    assert _host.group_quant(x, 128, 1e-10, False, False, False, False) is None
    assert _host.token_linear(x, w.t(), torch.ones(128), None, True) is None
    assert _host.block_linear(None, w, BLOCK, s, None) is None
    with FakeTensorMode():
        f = torch.empty((4, 256), dtype=torch.bfloat16, device="cuda")
        fw = torch.empty((128, 256), dtype=torch.float8_e4m3fn, device="cuda")
        assert _host.block_linear(f, fw, BLOCK, torch.empty((1, 2), device="cuda"), None) is None
        assert _host.group_quant(f, 128, 1e-10, False, False, False, False) is None


def test_declines_numbers_that_do_not_convert():
    """A number too large for the check is declined like any other, without an error left behind."""
    x, w, s = torch.zeros((4, 256), dtype=torch.bfloat16), torch.zeros((128, 256), dtype=torch.float8_e4m3fn), torch.ones((1, 2))
    assert _host.block_linear(x, w, [2**100, 128], s, None) is None
    with pytest.raises(RuntimeError, match="only block_size"):
        fp8_kernel.w8a8_block_fp8_matmul(w, w, s, s, [2**100, 128])


@pytest.fixture
def dispatcher(monkeypatch):
    """Calls fn() with every native call declining."""

    def call(fn):
        with monkeypatch.context() as m:
            for name in ("group_quant", "block_linear", "block_matmul", "token_linear", "mla_quant", "bmm", "fused_gate", "fused_experts"):
                assert hasattr(_host, name)
                m.setattr(_host, name, lambda *a: None)
            return fn()

    return call


def _same(a, b):
    if isinstance(a, tuple):
        return len(a) == len(b) and all(_same(x, y) for x, y in zip(a, b))
    if a.dtype == torch.float8_e4m3fn:
        a, b = a.view(torch.uint8), b.view(torch.uint8)
    return a.shape == b.shape and a.stride() == b.stride() and a.dtype == b.dtype and torch.equal(a, b)


def _randn(shape, dtype=torch.bfloat16, seed=0):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)).to(dtype).cuda()


def _weight(n, k, seed=1):
    return fp8_utils.per_block_cast_to_fp8(_randn((n, k), torch.float32, seed) * 0.02)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(1, 128, 128), (3, 264, 512), (33, 640, 1536), (300, 72, 256), (700, 1000, 384), (100, 1024, 4096),
                                   (1100, 4096, 256), (1300, 9224, 1024)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_linears_are_the_dispatcher_path(dev, dispatcher, m, n, k, dtype):
    x, (w, s), bias = _randn((m, k), dtype), _weight(n, k), _randn((n,), dtype, 2)
    for b in (None, bias):
        def block():
            return fp8_utils.w8a8_block_fp8_linear(x, w, BLOCK, s, bias=b)

        assert _host.block_linear(x, w, BLOCK, s, b) is not None
        assert _same(block(), dispatcher(block))
        for scale in (torch.rand((n, 1), device=dev) * 1e-2, torch.full((1,), 3e-3, device=dev)):
            def token():
                return fp8_utils.apply_fp8_linear(x, w.t(), scale, bias=b, use_per_token_if_dynamic=True)

            assert _host.token_linear(x, w.t(), scale, b, True) is not None
            assert _same(token(), dispatcher(token))
    q, xs = fp8_kernel.sglang_per_token_group_quant_fp8(x, 128)
    matmul = lambda: fp8_kernel.w8a8_block_fp8_matmul(q, w, xs, s, BLOCK, dtype)  # noqa: E731
    assert _same(matmul(), dispatcher(matmul))
    qp, xp = fp8_kernel.sglang_per_token_group_quant_fp8(x, 128, column_major_scales=True, scale_tma_aligned=True, scale_ue8m0=True)
    sgl_kernel.mark_ue8m0(s)
    packed = lambda: fp8_kernel.w8a8_block_fp8_matmul(qp, w, xp, s, BLOCK, dtype)  # noqa: E731
    assert (_host.block_matmul(qp, w, xp, s, BLOCK, dtype, True) is not None) == (m > 128)
    assert _same(packed(), dispatcher(packed))


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(1, 8, 128), (16, 136, 2048), (15, 1000, 128), (8, 4104, 4096), (7, 16376, 640), (1, 72, 18432), (2, 520, 8320),
                                   (1, 264, 32768), (3, 128, 10880)])
def test_quantising_decode_linear(dev, dispatcher, m, n, k):
    """One launch with the quantisation in it: smallest and largest activations it takes, rows of one to 256 groups, remainders of
    lane pieces, wave shares and weight rows, outliers, an all-zero row, a subnormal group scale; bit for bit the two launches."""
    from sglang_amd._lib import lib

    assert lib.fp8k_linear_fuses_quant(m, n, k) == 1
    assert lib.fp8k_linear_fuses_quant(32768 // k + 1, n, k) == 0 and lib.fp8k_linear_fuses_quant(17, n, k) == 0
    w, s = _weight(n, k)
    for dtype in (torch.bfloat16, torch.float16):
        x = _randn((m, k), dtype)
        x[:, ::97] *= 50
        x[m // 2, :128] *= 1e-7
        x[m - 1] = 0 if m > 1 else x[m - 1]
        for bias in (None, _randn((n,), dtype, 2), _randn((n,), torch.float32, 2)):
            calls = [lambda: fp8_utils.apply_fp8_linear(x, w.t(), torch.rand((n, 1), generator=torch.Generator().manual_seed(4)).to(dev),
                                                        bias=bias, use_per_token_if_dynamic=True)]
            if bias is None or bias.dtype == dtype:
                calls.append(lambda: fp8_utils.w8a8_block_fp8_linear(x, w, BLOCK, s, bias=bias))
            for call in calls:
                assert _same(call(), dispatcher(call))


@pytest.mark.gpu
@pytest.mark.parametrize("m,k", [(1, 128), (5, 640), (130, 7168)])
def test_group_quant_layouts_are_the_dispatcher_path(dev, dispatcher, m, k):
    x = _randn((m, k))
    for kw in ({}, dict(column_major_scales=True), dict(column_major_scales=True, scale_tma_aligned=True),
               dict(column_major_scales=True, scale_tma_aligned=True, scale_ue8m0=True), dict(fuse_silu_and_mul=True)):
        if k % 256 and "fuse_silu_and_mul" in kw:
            continue
        quant = lambda: fp8_kernel.sglang_per_token_group_quant_fp8(x, 128, **kw)  # noqa: E731
        assert _same(quant(), dispatcher(quant))


@pytest.mark.gpu
@pytest.mark.parametrize("heads,m,k,n", [(4, 1, 128, 512), (16, 37, 512, 128), (3, 130, 128, 264)])
def test_mla_products_are_the_dispatcher_path(dev, dispatcher, heads, m, k, n):
    x = _randn((m, heads, k)).transpose(0, 1)
    w, ws = fp8_utils.input_to_float8(_randn((heads, n, k), seed=3))

    def product():
        q, s = fp8_kernel.per_tensor_quant_mla_fp8(x, torch.zeros((1,), device=dev))
        return q, s, sgl_kernel.bmm_fp8(q, w.transpose(1, 2), s, ws, torch.bfloat16)

    assert _same(product(), dispatcher(product))


@pytest.mark.gpu
@pytest.mark.parametrize("heads,m,k", [(16, 17, 128), (5, 103, 72), (128, 64, 128), (64, 256, 128), (32, 512, 128), (32, 513, 128)])
def test_mla_quant_in_one_launch(dev, dispatcher, heads, m, k):
    """From one chunk of eight more than the one-workgroup form takes to one row more than the registers of the launch hold: the bytes
    and the scale of the two launches, in every one of a run of launches that share their counters, onto a scale that is not zero, on
    another stream and from a replayed graph in between."""
    x = _randn((m, heads, k)).transpose(0, 1)
    x[heads // 2, m // 3, k // 2] = 77

    def quant(start=0.0):
        return fp8_kernel.per_tensor_quant_mla_fp8(x, torch.full((1,), start, device=dev))

    for start in (0.0, 10.0):
        want = dispatcher(lambda: quant(start))
        assert all(_same(got, want) for got in [quant(start) for _ in range(20)])
    want = dispatcher(quant)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        outs = [quant() for _ in range(5)]
        side.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            captured = quant()
        for _ in range(3):
            graph.replay()
            outs.append(quant())
    torch.cuda.synchronize()
    assert all(_same(got, want) for got in outs + [captured])


@pytest.mark.gpu
def test_mla_quant_keeps_nothing_for_streams_from_outside(dev):
    """The counters of the one-launch form belong to a stream that torch made; under a handle that may come to mean another stream, or
    means one per thread, the two launches run."""
    x = _randn((64, 32, 128)).transpose(0, 1)
    want = fp8_kernel.per_tensor_quant_mla_fp8(x, torch.zeros((1,), device=dev))
    own, before = torch.cuda.Stream(), torch.cuda.memory_allocated()
    per_thread = 2  # hipStreamPerThread
    for stream in (torch.cuda.ExternalStream(own.cuda_stream), torch.cuda.ExternalStream(per_thread)):
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            got = fp8_kernel.per_tensor_quant_mla_fp8(x, torch.zeros((1,), device=dev))
        torch.cuda.synchronize()
        assert _same(got, want)
        del got
        assert torch.cuda.memory_allocated() == before


@pytest.mark.gpu
def test_mla_quant_in_one_launch_ends_its_wait(dev):
    """A count that never comes out (set from the host): every workgroup gives up its bounded wait and finds the maximum for itself."""
    from sglang_amd._lib import BF16, check, lib, stream_ptr

    x = _randn((40, 100, 128))
    want = fp8_kernel.per_tensor_quant_mla_fp8(x, torch.zeros((1,), device=dev))
    q, s = torch.empty_like(want[0]), torch.zeros((1,), device=dev)
    sync = torch.tensor([100000, 0, 0], dtype=torch.int32, device=dev)
    check(lib.fp8k_tensor_quant_mla_sync(x.data_ptr(), q.data_ptr(), s.data_ptr(), 40, 100, 128, x.stride(0), x.stride(1), 1e-12, BF16,
                                         sync.data_ptr(), stream_ptr(dev)))
    torch.cuda.synchronize()
    assert _same((q, s), want) and not sync.any()


@pytest.mark.gpu
def test_mla_quant_in_one_launch_waits_no_longer_than_it_saves(dev):
    """The largest tensor and a count that never comes out: 256 polls of 0.12 us and one workgroup's pass over 4 MB are 156 us (a wait
    of 4096 polls made it 576); twice that is allowed, for the median of 21."""
    from sglang_amd._lib import BF16, check, lib, stream_ptr

    x = _randn((32, 512, 128))
    q, times = torch.empty(x.shape, dtype=torch.float8_e4m3fn, device=dev), []
    for _ in range(21):
        s, sync = torch.zeros((1,), device=dev), torch.tensor([100000, 0, 0], dtype=torch.int32, device=dev)
        begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        begin.record()
        check(lib.fp8k_tensor_quant_mla_sync(x.data_ptr(), q.data_ptr(), s.data_ptr(), 32, 512, 128, x.stride(0), x.stride(1), 1e-12, BF16,
                                             sync.data_ptr(), stream_ptr(dev)))
        end.record()
        torch.cuda.synchronize()
        times.append(begin.elapsed_time(end) * 1e3)
    assert sorted(times)[10] < 312, times


@pytest.mark.gpu
@pytest.mark.parametrize("tokens", [1, 20, 100, 700])
def test_experts_are_the_dispatcher_path(dev, dispatcher, tokens):
    E, H, inter, topk = 16, 512, 256, 4
    x = _randn((tokens, H))
    parts = [[_weight(n, k, 10 * e + n) for e in range(E)] for n, k in ((2 * inter, H), (H, inter))]
    (w13, s13), (w2, s2) = [(torch.stack([q for q, _ in p]), torch.stack([s for _, s in p])) for p in parts]
    logits, bias = _randn((tokens, E), torch.float32, 7), _randn((E,), torch.float32, 8)

    def layer(inplace, on_input=False):
        tw, ids = fused_moe.biased_grouped_topk(x, logits, bias, topk, True, 4, 2)
        h = x.clone() if inplace else x
        out = fused_moe.fused_experts_impl(h, w13, w2, tw, ids, inplace=inplace, use_fp8_w8a8=True, w1_scale=s13, w2_scale=s2,
                                           block_shape=BLOCK, routed_scaling_factor=2.5, apply_router_weight_on_input=on_input)
        assert (out.data_ptr() == h.data_ptr()) == inplace
        return tw, ids, out

    for args in ((False,), (True,), (False, True)):
        assert _same(layer(*args), dispatcher(lambda: layer(*args)))


@pytest.mark.gpu
@pytest.mark.parametrize("inter", [256, 1024, 1152])
@pytest.mark.parametrize("tokens", [1, 3])
def test_experts_of_few_tokens_are_the_dispatcher_path(dev, dispatcher, tokens, inter):
    """Few blocks, up to, at and above the longest second K that takes the activation inside.  The largest terms of the second product
    cancel - its first K block against its last - so that another order of its sums shows in the 16-bit result."""
    E, H, topk = 16, 2048, 4
    x = _randn((tokens, H))
    g = torch.Generator().manual_seed(inter + tokens)
    fp8 = lambda t: t.to(dev).to(torch.float8_e4m3fn)  # noqa: E731
    w13, w2 = torch.randn((E, 2, inter, H), generator=g), torch.randn((E, H, inter), generator=g)
    w13[:, :, -128:] = w13[:, :, :128]
    w2[:, :, -128:] = -w2[:, :, :128]
    s13, s2 = torch.full((E, 2 * inter // 128, H // 128), 0.02), torch.rand((E, H // 128, inter // 128), generator=g) + 0.5
    s2[:, :, -1] = s2[:, :, 0] = 1000.0
    w13, w2, s13, s2 = fp8(w13.view(E, 2 * inter, H)), fp8(w2), s13.to(dev), s2.to(dev)
    logits, bias = _randn((tokens, E), torch.float32, 7), _randn((E,), torch.float32, 8)

    def layer():
        tw, ids = fused_moe.biased_grouped_topk(x, logits, bias, topk, True, 4, 2)
        return fused_moe.fused_experts_impl(x, w13, w2, tw, ids, use_fp8_w8a8=True, w1_scale=s13, w2_scale=s2, block_shape=BLOCK,
                                            routed_scaling_factor=2.5)

    assert _same(layer(), dispatcher(layer))


@pytest.mark.gpu
@pytest.mark.parametrize("b,m,n,k", [(1, 1, 8, 128), (9, 64, 128, 256), (8, 65, 136, 384), (17, 127, 120, 1024), (3, 70, 200, 1152)])
def test_bmm_tile_edges(dev, b, m, n, k):
    """Row, column and batch remainders of the short-K kernel's 64 x 128 tiles, one to nine K blocks, strided operands and
    output; exact on integer data."""
    g = torch.Generator().manual_seed(m)
    A = torch.randint(-4, 5, (b, m + 3, k), generator=g).float()
    B = torch.randint(-4, 5, (b, n, k), generator=g).float()
    out = torch.zeros((b, m + 1, n + 8), dtype=torch.float16, device=dev)
    fa, fb = A.to(dev).to(torch.float8_e4m3fn), B.to(dev).to(torch.float8_e4m3fn)
    one = torch.ones((1,), device=dev)
    sgl_kernel.bmm_fp8(fa[:, :m], fb.transpose(1, 2), one * 0.5, one * 0.25, torch.float16, out[:, :m, :n])
    ref = (A[:, :m] @ B.transpose(1, 2)) * 0.125
    assert torch.equal(out[:, :m, :n].float().cpu(), ref.half().float())
    assert not out[:, m:].any() and not out[:, :, n:].any()


def _calls(dev):
    """One call per native function, of arguments it takes."""
    x, (w, s) = _randn((40, 512)), _weight(256, 512)
    q, xs = fp8_kernel.sglang_per_token_group_quant_fp8(x, 128)
    h, e = _randn((20, 4, 128)).transpose(0, 1), 8
    wb, wbs = fp8_utils.input_to_float8(_randn((4, 256, 128), seed=3))
    qh, hs = fp8_kernel.per_tensor_quant_mla_fp8(h, torch.zeros((1,), device=dev))
    logits, bias = _randn((40, e), torch.float32), _randn((e,), torch.float32)
    tw, ids = fused_moe.biased_grouped_topk(x, logits, bias, 2, True, 4, 2)
    w13, s13 = w.repeat(e, 1, 1).contiguous(), s.repeat(e, 1, 1).contiguous()
    w2, s2 = [t.repeat(e, 1, 1).contiguous() for t in _weight(512, 128)]
    return {
        "group_quant": (x, 128, 1e-10, False, False, False, False),
        "block_linear": (x, w, BLOCK, s, None),
        "block_matmul": (q, w, xs, s, BLOCK, torch.bfloat16, False),
        "token_linear": (x, w.t(), torch.ones((256, 1), device=dev), None, True),
        "mla_quant": (h, torch.zeros((1,), device=dev), 1e-12),
        "bmm": (qh, wb.transpose(1, 2), hs, wbs, torch.bfloat16),
        "fused_gate": (logits, bias, 4, 2, 2, 0, 0.0, False),
        "fused_experts": (x, w13, w2, s13, s2, tw, ids, 16, False, False, False, 1.0, False),
    }


@pytest.mark.gpu
def test_other_threads_run_during_the_calls(dev):
    """With a switch interval that nothing here reaches, another thread gets the interpreter only where a call gives it up."""
    calls, ticks, stop = _calls(dev), [0], threading.Event()

    def count():
        while not stop.is_set():
            ticks[0] += 1
            time.sleep(0)

    thread, interval = threading.Thread(target=count), sys.getswitchinterval()
    sys.setswitchinterval(60.0)
    try:
        thread.start()
        for name, args in calls.items():
            fn, results, before = getattr(_host, name), [], ticks[0]  # kept: freeing a tensor gives the interpreter up as well
            while len(results) < 5000 and ticks[0] == before:
                results.append(fn(*args))
            assert ticks[0] != before and all(r is not None for r in results), name
    finally:
        stop.set()
        sys.setswitchinterval(interval)
        thread.join()
    torch.cuda.synchronize()


class _Sub(torch.Tensor):
    """A subclass without __torch_dispatch__: its key set is that of a plain tensor."""


class _Quiet(torch.Tensor):
    __torch_function__ = torch._C._disabled_torch_function_impl


class _Record(TorchFunctionMode):
    def __init__(self):
        super().__init__()
        self.seen = []

    def __torch_function__(self, func, types, args=(), kwargs=None):
        self.seen.append(str(func))
        return func(*args, **(kwargs or {}))


@pytest.mark.gpu
def test_function_subclasses_and_modes_are_seen(dev, dispatcher):
    """Every native call declines a tensor of a class with a __torch_function__, in any place, and all of them under a function
    mode; parameters and classes that switch theirs off are taken."""
    for name, args in _calls(dev).items():
        fn, places = getattr(_host, name), [i for i, a in enumerate(args) if isinstance(a, torch.Tensor)]

        def with_class(i, cls):
            return [a.as_subclass(cls) if j == i else a for j, a in enumerate(args)]

        for i in places:
            assert fn(*with_class(i, _Sub)) is None, (name, i)
            assert fn(*with_class(i, _Quiet)) is not None, (name, i)
            if args[i].is_floating_point() and args[i].element_size() > 1:
                param = [torch.nn.Parameter(a, requires_grad=False) if j == i else a for j, a in enumerate(args)]
                assert fn(*param) is not None, (name, i)
        with torch._C.DisableTorchFunctionSubclass():
            assert fn(*with_class(places[0], _Sub)) is not None
        with _Record():
            assert fn(*args) is None, name
    # through the entry points: what comes back and what a mode sees are the dispatcher path's
    x, (w, s) = _randn((40, 512)), _weight(256, 512)
    sub = x.as_subclass(_Sub)
    for call in (lambda: fp8_utils.w8a8_block_fp8_linear(sub, w, BLOCK, s),
                 lambda: fp8_utils.w8a8_block_fp8_linear(x, w.as_subclass(_Sub), BLOCK, s),
                 lambda: fp8_utils.apply_fp8_linear(sub, w.t(), torch.ones((256, 1), device=dev), use_per_token_if_dynamic=True),
                 lambda: fp8_kernel.sglang_per_token_group_quant_fp8(sub, 128)[0]):
        got, want = call(), dispatcher(call)
        assert type(got) is type(want) and _same(got.as_subclass(torch.Tensor), want.as_subclass(torch.Tensor))
        seen = []
        for run in (call, lambda: dispatcher(call)):
            with _Record() as mode:
                run()
            seen.append(mode.seen)
        assert seen[0] == seen[1] and any("fp8k" in f for f in seen[0])


@pytest.mark.gpu
def test_profiler_sees_the_calls(dev):
    """A record per native call, with the shapes of its tensors, where the dispatcher keeps one of an op."""
    calls = _calls(dev)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU], record_shapes=True) as prof:
        for name, args in calls.items():
            getattr(_host, name)(*args)
    records = {e.name: e for e in prof.events() if e.name.startswith("fp8k::")}
    assert set(records) == {"fp8k::" + name for name in calls}
    for name, args in calls.items():
        shapes = [list(a.shape) for a in args if isinstance(a, torch.Tensor) and a.dim()]
        assert [s for s in records["fp8k::" + name].input_shapes if s] == shapes, name


@pytest.mark.gpu
def test_threads_that_share_a_stream_share_its_workspace(dev):
    """Products with K cut through float partials, of two threads on one stream at once: the launches of one do not come between
    those of the other."""
    from sglang_amd._lib import lib

    m, n, k = 128, 1024, 8192
    assert lib.fp8k_block_gemm_workspace_bytes(m, n, k) > m * n * 8  # partials of two and more K ranges
    w, s = _weight(n, k)
    jobs = [fp8_kernel.sglang_per_token_group_quant_fp8(_randn((m, k), seed=seed), 128, column_major_scales=True) for seed in (1, 2)]
    want = [fp8_kernel.w8a8_block_fp8_matmul(q, w, xs, s, BLOCK, torch.bfloat16) for q, xs in jobs]
    torch.cuda.synchronize()
    got, start = [None, None], threading.Barrier(2)

    def work(i):
        q, xs = jobs[i]
        start.wait()
        got[i] = [_host.block_matmul(q, w, xs, s, BLOCK, torch.bfloat16, False) for _ in range(500)]

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for i in range(2):
        assert all(torch.equal(out, want[i]) for out in got[i])


@pytest.mark.parametrize("held", [0, 1 << 20])
@pytest.mark.parametrize("needs", [(40 << 20, 40 << 20), (40 << 20, 100 << 20)])
def test_no_workspace_handed_out_is_released(monkeypatch, held, needs):
    """Threads that first need, or outgrow, the workspace of one stream at the same moment: what each of them is given is large
    enough and stays alive, in use or retired."""
    buffers, retired, real = {}, [], torch.empty
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device: types.SimpleNamespace(cuda_stream=7))
    if held:
        buffers[None, 7] = real(held, dtype=torch.uint8)
    monkeypatch.setattr(sgl_kernel, "_workspaces", buffers)
    monkeypatch.setattr(sgl_kernel, "_retired", retired)
    met = threading.Barrier(2)

    def empty(*args, **kwargs):
        met.wait(timeout=30)  # neither thread has stored its buffer when the other has decided to make one
        return real(*args, **kwargs)

    monkeypatch.setattr(torch, "empty", empty)
    got = [None, None]

    def work(i):
        got[i] = sgl_kernel._workspace(torch.device("cpu"), needs[i])

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    kept = [*buffers.values(), *retired]
    for buf, need in zip(got, needs):
        assert buf.numel() >= need and any(buf is k for k in kept)
    assert len({id(k) for k in kept}) == len(kept)
    assert buffers[None, 7].numel() >= max(needs)
