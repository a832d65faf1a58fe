"""Dynamically quantized linears of up to 16 rows in one launch (csrc/few_rows.hip): the bits of the row quantizer followed by the product."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.float16, torch.bfloat16]
# (rows, k, n): the smallest; K of part steps and part segments; one, two and four segments a wavefront and 1 .. 4 steps, at their edges;
# part blocks of channels, one, two and four blocks a workgroup
INT8 = [(1, 16, 1), (3, 272, 100), (16, 512, 17), (16, 1024, 1024), (15, 1520, 33), (10, 1040, 33), (2, 8192, 16), (1, 6160, 40), (4, 4096, 4096), (16, 2048, 4097), (5, 640, 16400)]
TERNARY = [(2, 64, 1), (16, 64, 300), (7, 1088, 72), (16, 2048, 2049), (4, 8192, 36), (3, 4096, 8192), (1, 4096, 8192), (8, 3648, 5)]


def rows_of(case, m, k, dtype, gen):
    x = torch.randn(m, k, device="cuda", generator=gen)
    if case == 1:  # below eps, zeros, an infinity, a NaN, the maximum in the last element
        x[0] *= 1e-7
        x[m // 2] *= 0.0
        x[m - 1, k - 1] = -300.0
    if case == 2:
        x[0, k // 2] = float("inf")
        x[m - 1, 0] = float("nan")
    return x.to(dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m,k,n", INT8)
def test_int8_rows_quantized_in_the_product(m, k, n, dtype):
    from tensorplay_amd import _lib, ops

    gen = torch.Generator(device="cuda").manual_seed(m + k + n)
    lib = _lib.load()
    w = torch.randint(-128, 128, (n, k), device="cuda", generator=gen, dtype=torch.int8)
    scale, bias = torch.rand(n, device="cuda", generator=gen), torch.randn(n, device="cuda", generator=gen)
    for case in range(3):
        x = rows_of(case, m, k, dtype, gen)
        assert lib.tpq_int8_linear_few_takes(x.data_ptr(), w.data_ptr(), m, n, k) == 1
        codes, row_scale = ops._quantize_int8_rowwise(x, 1e-5)
        for b, out_dtype in ((None, dtype), (bias, torch.float32)):
            want = ops.int8_mm_dequant(codes, w, row_scale, scale, bias=b, out_dtype=out_dtype)
            got = torch.empty(m, n, device="cuda", dtype=out_dtype)
            ops._check(lib.tpq_int8_linear_few(x.data_ptr(), ops._DT[dtype], w.data_ptr(), scale.data_ptr(), ops._ptr(b), m, n, k, 1e-5, got.data_ptr(),
                                               ops._DT[out_dtype], ops._stream(x)))
            assert torch.equal(got.view(torch.uint8), want.view(torch.uint8)), (case, b is not None)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m,k,n", TERNARY)
def test_ternary_rows_quantized_in_the_product(m, k, n, dtype):
    from tensorplay_amd import _lib, ops

    gen = torch.Generator(device="cuda").manual_seed(m + k + n)
    lib = _lib.load()
    packed = ops.pack_ternary(torch.randint(-1, 2, (n, k), device="cuda", generator=gen, dtype=torch.int8))
    bias = torch.randn(n, device="cuda", generator=gen)
    for case in range(3):
        x = rows_of(case, m, k, dtype, gen)
        assert lib.tpq_ternary_linear_few_takes(x.data_ptr(), packed.data_ptr(), m, n, k) == 1
        codes, row_scale = ops._quantize_int8_rowwise(x, 1e-5)
        for b in (None, bias):
            want = ops.ternary_mm(codes, row_scale, packed, 0.037, k, bias=b)
            assert torch.equal(ops._ternary_linear(x, packed, 0.037, k, b, 1e-5).view(torch.int32), want.view(torch.int32)), (case, b is not None)


def test_the_rule_of_the_one_launch_linears():
    """What is refused goes to the two launches: rows, K, weight and alignment on both sides of the line."""
    from tensorplay_amd import _lib

    lib = _lib.load()

    def int8(m, k, n, at=4096):
        return lib.tpq_int8_linear_few_takes(at, 4096, m, n, k)

    def ternary(m, k, n, at=4096):
        return lib.tpq_ternary_linear_few_takes(at, 4096, m, n, k)

    assert (int8(16, 1024, 64), int8(17, 1024, 64), int8(0, 1024, 64)) == (1, 0, 0)
    assert (int8(1, 1024, 64, 4100), int8(1, 1032, 64), int8(1, 8192, 64), int8(1, 8208, 64)) == (0, 0, 1, 0)
    assert (int8(16, 2048, 4096), int8(16, 2064, 4096), int8(7, 3328, 1280), int8(4, 8192, 1024)) == (1, 0, 0, 0)
    assert (int8(1, 4096, 8192), int8(1, 4096, 8193), int8(1, 512, 32768), int8(1, 512, 32769)) == (1, 0, 1, 0)
    assert (ternary(16, 2048, 64), ternary(16, 2112, 64), ternary(1, 96, 64), ternary(16, 64, 64, 4104)) == (1, 0, 0, 0)


def test_linears_on_both_sides_of_the_line_in_a_graph():
    """The modules' calls, eager and captured, replayed with new inputs."""
    from tensorplay_amd import ops
    from tensorplay_amd.ao import quantization as q

    gen = torch.Generator(device="cuda").manual_seed(5)
    for rows in (16, 17):
        lin = torch.nn.Linear(1024, 520, device="cuda", dtype=torch.float16)
        module = q.Int8DynamicLinear.from_float(lin, out_dtype=torch.float16)
        x = torch.randn(rows, 1024, device="cuda", generator=gen).half()
        module(x)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = module(x)
        for _ in range(3):
            x.copy_(torch.randn(rows, 1024, device="cuda", generator=gen))
            graph.replay()
            codes, scale = ops._quantize_int8_rowwise(x, 1e-5)
            want = ops.int8_mm_dequant(codes, module.weight, scale, module.weight_scale, bias=module.bias, out_dtype=torch.float16)
            assert torch.equal(out, want) and torch.equal(module(x), want)


# (kind, rows, k, n): where the one launch is the longer one on the device and on both sides of that line
PAYS = [("int8", 8, 4096, 4096, 1), ("int8", 11, 2528, 2460, 1), ("int8", 16, 1984, 2272, 1), ("int8", 12, 1984, 2272, 2), ("int8", 2, 4096, 4096, 2), ("int8", 1, 7392, 1348, 0),
        ("int8", 1, 7424, 1348, 2), ("int8", 3, 4272, 924, 1), ("int8", 3, 4288, 924, 2), ("int8", 17, 1024, 64, 0), ("ternary", 16, 2048, 2048, 1), ("ternary", 16, 1984, 2048, 2),
        ("ternary", 8, 2048, 2048, 2)]


@pytest.mark.parametrize("kind,m,k,n,pays", PAYS)
def test_one_launch_where_it_pays(kind, m, k, n, pays):
    """Eager calls save a launch and its buffer wherever the device is not longer by more; a captured call takes the shorter way on the device.  The same
    bits either way, eager, captured and replayed; the way shows in the allocations (the result, and the codes that two launches need)."""
    from tensorplay_amd import _lib, ops
    from tensorplay_amd.ao import quantization as q

    lib = _lib.load()
    assert (lib.tpq_int8_linear_few_pays if kind == "int8" else lib.tpq_ternary_linear_few_pays)(m, n, k) == pays
    lin = torch.nn.Linear(k, n, bias=False, device="cuda", dtype=torch.float16)
    module = q.Int8DynamicLinear.from_float(lin, out_dtype=torch.float16) if kind == "int8" else q.BitNetPacked2bitLinear.from_float(lin)
    gen = torch.Generator(device="cuda").manual_seed(m + k + n)
    x = torch.randn(m, k, device="cuda", generator=gen).half()

    def codes_and_product():
        codes, scale = ops._quantize_int8_rowwise(x, 1e-5)
        if kind == "int8":
            return ops.int8_mm_dequant(codes, module.weight, scale, module.weight_scale, bias=module.bias, out_dtype=torch.float16)
        return ops.ternary_mm(codes, scale, module.int_data, float(module.scale), k, bias=module.bias)

    def allocations(call):
        before = torch.cuda.memory_stats()["allocation.all.allocated"]
        out = call()
        return out, torch.cuda.memory_stats()["allocation.all.allocated"] - before

    with torch.no_grad():
        module(x)
        torch.cuda.synchronize()
        _, eager = allocations(lambda: module(x))
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out, captured = allocations(lambda: module(x))
        assert (eager > 1, captured > 1) == (pays == 0, pays < 2)
        for _ in range(3):
            x.copy_(torch.randn(m, k, device="cuda", generator=gen))
            graph.replay()
            want = codes_and_product()
            assert torch.equal(out, want) and torch.equal(module(x), want)
