"""GPU parity: fused row-wise quantizer vs the CPU oracle, bit-exact codes and scales."""
import numpy as np
import pytest
import torch

import oracle
from gpu_util import DEV, cast_bits, dev, host

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from tensorplay_amd import ops as _ops

    return _ops


SHAPES = [(1, 1), (3, 5), (16, 1024), (7, 2560), (1, 6912), (5, 4099), (4, 8), (2, 16384), (2, 20000),
          (3, 16392), (128, 6912), (300, 2048), (2048, 4096),
          (1000, 64), (77, 56), (33, 128), (5, 200), (129, 512), (9, 264), (70, 1000), (4097, 1024), (3, 1032),
          (3, 28672), (2, 65536), (2, 65544), (5, 40000)]


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("shape", SHAPES)
def test_int8_rowwise_bit_exact(ops, dtype, shape):
    rng = np.random.default_rng(shape[0] * 7919 + shape[1])
    x = rng.normal(size=shape).astype(np.float32)
    if shape[0] > 2:
        x[1] = 0.0                       # all-zero row: scale = eps / 127, codes 0
        x[2] *= 1e-7                     # below eps
    if shape == (2048, 4096):            # outlier columns of the prefill configuration
        x[:, rng.choice(4096, 41, replace=False)] *= 20.0
    xb = cast_bits(x, dtype)
    want_codes, want_scales = oracle.quantize_int8_rowwise(xb, dtype, 1e-5)
    codes, scales = ops._quantize_int8_rowwise(dev(xb, dtype), 1e-5)
    assert codes.dtype == torch.int8 and scales.dtype == torch.float32 and scales.shape == (shape[0],)
    np.testing.assert_array_equal(host(scales), want_scales)
    np.testing.assert_array_equal(host(codes), want_codes)


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("k", [4, 12, 20, 60, 68, 132, 260, 516, 1020, 1028, 2044, 2052, 5284, 16388, 65532])
def test_rows_of_fours_bit_exact(ops, dtype, k):
    """K % 8 == 4: the last eight elements of a row overlap the chunk before them, and rows start on 8 bytes; the row maximum in
    the last four, in the overlap and in the first element."""
    rng = np.random.default_rng(k)
    x = rng.normal(size=(5, k)).astype(np.float32)
    for row, at in ((0, k - 1), (1, max(k - 8, 0)), (2, 0), (3, k // 2)):
        x[row, at] = -9.0
    xb = cast_bits(x, dtype)
    want_codes, want_scales = oracle.quantize_int8_rowwise(xb, dtype, 1e-5)
    codes, scales = ops._quantize_int8_rowwise(dev(xb, dtype), 1e-5)
    np.testing.assert_array_equal(host(scales), want_scales)
    np.testing.assert_array_equal(host(codes), want_codes)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_lowbit_variants_bit_exact(ops, dtype):
    rng = np.random.default_rng(5)
    x = rng.normal(size=(37, 1000)).astype(np.float32)
    x[3, :5] = [0.5, 1.5, 2.5, -0.5, -1.5]
    xb = cast_bits(x, dtype)
    xd = dev(xb, dtype)
    for fn, ofn in ((ops._quantize_int4_rowwise, oracle.quantize_int4_rowwise),
                    (ops._quantize_int2_rowwise, oracle.quantize_int2_rowwise),
                    (ops._quantize_binary_rowwise, oracle.quantize_binary_rowwise)):
        c, s = fn(xd, 1e-8)
        wc, ws = ofn(xb, dtype, 1e-8)
        np.testing.assert_array_equal(host(c), wc)
        np.testing.assert_array_equal(host(s), ws)


def test_ties_round_to_even(ops):
    x = torch.tensor([[127, -127, 0.5, 1.5, 2.5, -0.5, -1.5, -2.5]], device=DEV)
    codes, scales = ops._quantize_int8_rowwise(x, 1e-5)
    assert scales.item() == 1.0
    assert codes.cpu().tolist() == [[127, -127, 0, 2, 2, 0, -2, -2]]


def test_non_contiguous_and_empty_and_errors(ops):
    x = torch.randn(64, 96, device=DEV)
    view = x[:, ::2]
    c, s = ops._quantize_int8_rowwise(view, 1e-5)
    wc, ws = oracle.quantize_int8_rowwise(view.cpu().contiguous().numpy())
    np.testing.assert_array_equal(host(c), wc)
    np.testing.assert_array_equal(host(s), ws)
    c, s = ops._quantize_int8_rowwise(torch.empty(0, 8, device=DEV), 1e-5)
    assert c.shape == (0, 8) and s.shape == (0,)
    with pytest.raises(ValueError):
        ops._quantize_int8_rowwise(torch.zeros(2, 2, 2, device=DEV), 1e-5)
    with pytest.raises(TypeError):
        ops._quantize_int8_rowwise(torch.zeros(2, 2, device=DEV, dtype=torch.float64), 1e-5)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,k,n", [
    # rows read as they are and padded to 128; one, two, four and eight chunks of the quantizer at their edges; the longest row and one beyond
    (40, 16, 9), (33, 2048, 70), (5, 2052, 33), (129, 4096, 65), (36, 4100, 40), (3, 8188, 17), (2, 16384, 5), (34, 16388, 6),
    # the shortest row, a row below it, rows that are no multiple of four
    (40, 8, 5), (40, 4, 5), (35, 1023, 24), (300, 808, 256)])
def test_both_operands_prepared_in_one_launch(m, k, n, dtype):
    """The quantizer of the activations beside that of the weight (training linears) or the copy of an int8 weight to padded rows: the
    bits of the separate operators, for ordinary rows and for ones that are zero, tiny, infinite or NaN, several calls one after another."""
    from tensorplay_amd import ops
    from tensorplay_amd.ao.quantization import int8_dyn_act_lowbit as low

    gen = torch.Generator(device="cuda").manual_seed(m + k + n)
    x, w = (torch.randn(r, k, device="cuda", generator=gen) for r in (m, n))
    for a in (x, w):
        a[0] = 0.0
        a[1] *= 1e-9
        a[-1, k // 2] = -300.0
    x[m // 2, k - 1] = float("inf")
    w[n // 2, 0] = float("nan")
    x, w = x.to(dtype), w.to(dtype)
    codes, scale = ops._quantize_int8_rowwise(x, 1e-5)
    for quantize in (low._quantize_int4_weight_signed, low._quantize_int2_weight_signed, low._quantize_binary_weight_signed):
        w_codes, w_scale = quantize(w)
        want = ops.int8_mm_dequant(codes, w_codes, scale, w_scale)
        got = low._Int8DynActLowBitLinear.apply(x, w, quantize)
        assert torch.equal(got.view(torch.int32), want.view(torch.int32))
    w8, w_scale = ops._quantize_int8_rowwise(torch.randn(n, k, device="cuda", generator=gen), 1e-5)
    bias = torch.randn(n, device="cuda", generator=gen)
    for b in (None, bias, None):
        want = ops.int8_mm_dequant(codes, w8, scale, w_scale, b, torch.float32)
        got = ops._int8_dynamic_linear(x, w8, w_scale, b, torch.float32)
        assert torch.equal(got.view(torch.int32), want.view(torch.int32))
