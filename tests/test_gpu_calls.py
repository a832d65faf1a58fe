"""The native calls behind the hot operators against the operators' Python form: the same bits for operands of every form that
either takes, and the same refusals."""
import pytest
import torch

from tensorplay_amd import _lib, ops
from tensorplay_amd.ao import quantization as q

pytestmark = pytest.mark.gpu

DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def _shifted(x):
    """The same values one element off the allocation's alignment."""
    buf = torch.empty(x.numel() + 1, dtype=x.dtype, device=x.device)
    buf[1:].copy_(x.reshape(-1))
    return buf[1:].view(x.shape)


def _forms(x):
    yield x
    yield x.view(1, *x.shape)
    yield torch.cat([x, x], 1)[:, : x.shape[1]]   # rows apart
    yield x.t().contiguous().t()
    yield _shifted(x)
    yield x.clone().requires_grad_()
    yield x[:0]


def _both(monkeypatch, call):
    lib = _lib.load()
    with torch.no_grad():
        native = call()
    with monkeypatch.context() as patch:
        patch.setattr(lib, "calls", None)
        with torch.no_grad():
            plain = call()
    return native, plain


def _same(a, b):
    if isinstance(a, ops.PackedCodes):
        assert a.shape == b.shape and a.dtype == b.dtype
        a, b = a.data, b.data
    assert a.shape == b.shape and a.dtype == b.dtype and a.is_contiguous() == b.is_contiguous()
    assert torch.equal(a.view(torch.uint8) if a.numel() else a, b.view(torch.uint8) if b.numel() else b)


def _module(kind, k, n, dtype, bias):
    lin = torch.nn.Linear(k, n, bias=bias, device="cuda", dtype=dtype)
    if kind == "int8":
        return q.Int8DynamicLinear.from_float(lin, out_dtype=dtype)
    if kind == "int4":
        return q.WeightOnlyInt4Linear.from_float(lin, 64)
    if kind == "intx":
        return q.WeightOnlyIntxLinear.from_float(lin, bits=2, groupsize=64)
    return q.BitNetPacked2bitLinear.from_float(lin)


@pytest.mark.parametrize("kind", ["int8", "int4", "intx", "bitnet"])
@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("rows", [1, 16, 17, 40])
def test_modules(monkeypatch, kind, dtype, rows):
    gen = torch.Generator(device="cuda").manual_seed(rows)
    # 192: a K that no 128-wide kernel takes whole; 4 more for the kernels that want nothing of K
    # 4096 against few channels: slices of K, whose second kernel adds the bias
    for k, n, bias in ((512, 200, True), (4096, 72, True), (192, 72, False), *(((196, 72, False),) if kind in ("int8", "bitnet") else ())):
        module = _module(kind, k, n, DTYPES[dtype], bias)
        x = torch.randn(rows, k, device="cuda", generator=gen).to(DTYPES[dtype])
        for form in _forms(x):
            _same(*_both(monkeypatch, lambda: module(form)))


def test_int4_off_alignment_takes_any_address(monkeypatch):
    """Rows that start at any element are taken whatever the row count, as with one row."""
    module = _module("int4", 512, 256, torch.float16, False)
    x = torch.randn(40, 512, device="cuda", dtype=torch.float16)
    want = module(x).float()
    got = module(_shifted(x)).float()
    # both round float32 sums once to float16 (the other kernel also each weight product): a few units in the last place of the largest
    assert (got - want).abs().max() <= 4e-3 * want.abs().max()
    intx = _module("intx", 512, 256, torch.float32, False)
    x = torch.randn(24, 512, device="cuda")
    assert (intx(_shifted(x)) - intx(x)).abs().max() <= 1e-5 * intx(x).abs().max()


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("storage", ["quint4x2", "qint8", "quint2x4", "quint1x8", "qint32"])
def test_affine_codec(monkeypatch, dtype, storage):
    least, most = {"quint4x2": (0, 15), "qint8": (-128, 127), "quint2x4": (0, 3), "quint1x8": (0, 1), "qint32": (-1000, 1000)}[storage]
    x = torch.randn(24, 96, device="cuda").to(DTYPES[dtype])
    scale = torch.rand(24, 3, device="cuda") + 0.01
    zero = torch.randint(least, most + 1, (24, 3), device="cuda").float()
    for zp in (zero, None, zero.to(torch.float64)):
        for form in (x, _shifted(x), x.t().contiguous().t()):
            for block in ((1, 32), [1, 32]):
                codes = _both(monkeypatch, lambda: ops.quantize_affine(form, block, scale, zp, storage, least, most))
                _same(*codes)
                _same(*_both(monkeypatch, lambda: ops.dequantize_affine(codes[0], block, scale, zp)))


def test_refusals_are_the_python_forms():
    x = torch.randn(4, 512, device="cuda", dtype=torch.float16)
    module = _module("int4", 512, 256, torch.float16, False)
    with pytest.raises(ValueError):
        ops._weight_int4pack_mm(x[0], module.weight, 64, module.scales_and_zeros)
    with pytest.raises(ValueError):
        ops._weight_int4pack_mm(x, module.weight, 48, module.scales_and_zeros)
    with pytest.raises(ValueError):
        ops._weight_int4pack_mm(x[:, :480], module.weight, 64, module.scales_and_zeros)
    with pytest.raises(RuntimeError):
        ops._quantize_int8_rowwise(x.cpu(), 1e-5)
    with pytest.raises(TypeError):
        ops._quantize_int8_rowwise(x.double(), 1e-5)
    codes, scales = ops._quantize_int8_rowwise(x, 1e-5)
    with pytest.raises(ValueError):
        ops.int8_mm_dequant(codes, codes, scales[:2], scales)
    with pytest.raises(ValueError):
        ops.quantize_affine(x, (1, 512, 1), scales, None, "qint8", -128, 127)
    with pytest.raises(ValueError):
        ops.quantize_affine(x, (1, 512), scales[:3], None, "qint8", -128, 127)


def test_modes_and_transforms_see_the_python_form():
    from torch.utils._python_dispatch import TorchDispatchMode

    class Count(TorchDispatchMode):
        seen = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            Count.seen += 1
            return func(*args, **(kwargs or {}))

    module = _module("int8", 512, 256, torch.float16, False)
    x = torch.randn(4, 512, device="cuda", dtype=torch.float16)
    want = module(x)
    with Count():
        got = module(x)
    assert Count.seen > 0 and torch.equal(got, want)


def test_streams_and_graph():
    """On a side stream, and replayed from a graph with new inputs, with eager work between the replays."""
    module = _module("int4", 4096, 256, torch.bfloat16, True)
    int8 = _module("int8", 4096, 256, torch.bfloat16, True)
    x = torch.randn(40, 4096, device="cuda", dtype=torch.bfloat16)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        first = module(x), int8(x)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        outs = module(x), int8(x)
    for step in range(3):
        if step:
            x.copy_(torch.randn(40, 4096, device="cuda"))
        graph.replay()
        torch.cuda.synchronize()
        want = module(x), int8(x)
        torch.cuda.synchronize()
        assert torch.equal(outs[0], want[0]) and torch.equal(outs[1], want[1])
        if not step:
            assert torch.equal(first[0], want[0]) and torch.equal(first[1], want[1])


def test_int4_workspace_lives_until_the_launch():
    """Another thread may replace the stream's workspace while a call is without the GIL: the call's own stays alive until its
    kernel is enqueued.  The replacement happens where the call allocates its result (the allocator reports every allocation)."""
    import weakref

    from torch.cuda import _gpu_trace

    module = q.WeightOnlyInt4Linear.from_float(torch.nn.Linear(4096, 264, bias=False, device="cuda", dtype=torch.float16), 128)
    x = torch.randn(8, 4096, device="cuda", dtype=torch.float16)
    with torch.no_grad():
        want = module(x)
    key = (torch.cuda.current_device(), torch.cuda.current_stream().cuda_stream)
    held = weakref.ref(ops._int4_workspaces[key])
    larger = torch.zeros(ops._int4_workspaces[key].numel() + 4096, dtype=torch.uint8, device="cuda")
    seen = []

    def replace(_):
        if not seen:
            ops._int4_workspaces[key] = larger
            seen.append(held() is not None)

    callbacks = _gpu_trace.MemoryAllocationCallbacks
    torch._C._activate_gpu_trace()
    callbacks.add_callback(replace)
    try:
        with torch.no_grad():
            got = module(x)
    finally:
        callbacks.callback_list.remove(replace)
    assert seen == [True] and torch.equal(got, want)
    with torch.no_grad():
        assert torch.equal(module(x), want)
    assert held() is None  # and no longer


def test_refused_before_anything_is_allocated():
    """Operands that the fused launches do not take: the native call returns to the Python form with nothing allocated."""
    calls = _lib.load().calls
    x = {k: torch.randn(48, k, device="cuda") for k in (516, 518, 16388, 4)}
    w8 = {k: torch.ones(64, k, dtype=torch.int8, device="cuda") for k in x}
    w = {k: torch.randn(64, k, device="cuda") for k in x}
    scale, grad, few = torch.ones(64, device="cuda"), torch.randn(48, 64, device="cuda"), torch.randn(3, 64, device="cuda")
    shifted = {k: _shifted(v) for k, v in x.items()}
    before = torch.cuda.memory_stats()["allocation.all.allocated"]
    for k in (518, 16388, 4):  # K % 4, above 16384 with K % 16, below 8
        assert calls.int8_linear(x[k], w8[k], scale, None, 1e-5, torch.float32, 32) is None
        assert calls.lowbit_linear(x[k], w[k], 1e-5, 1e-8, 7.0, -8, 7, 0) is None
    assert calls.lowbit_linear(shifted[516], w[516], 1e-5, 1e-8, 7.0, -8, 7, 0) is None
    with torch.no_grad():
        assert calls.linear_grads(grad, x[518], w[518], True, True) is None
        assert calls.linear_grads(grad, shifted[516], w[516], True, True) is None
        assert calls.linear_grads(few, x[516][:3], w[516], True, True) is None  # up to three rows the products are the faster ones
    assert torch.cuda.memory_stats()["allocation.all.allocated"] == before


def test_a_full_card_leaves_the_routes_with_less_memory():
    """Where the memory for the weight written out as int8 is not there, the kernels of the packed weight run, which need none."""
    torch.manual_seed(0)
    lin = _module("bitnet", 8192, 28672, torch.bfloat16, False)  # a workspace of 235 MB from 257 rows on
    x = torch.randn(260, 8192, device="cuda", dtype=torch.bfloat16)
    with torch.no_grad():
        want = lin(x)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    try:
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (120 << 20)) / total)
        with torch.no_grad():
            assert torch.equal(lin(x), want)
            torch.cuda.empty_cache()
            taken = []
            with pytest.raises(torch.OutOfMemoryError):  # (64 of 8 MB are far more than is allowed)
                for _ in range(64):
                    taken.append(torch.empty(8 << 20, dtype=torch.uint8, device="cuda"))
            with pytest.raises(torch.OutOfMemoryError):
                lin(x)  # nothing left for the result, of 30 MB, either
            del taken
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
