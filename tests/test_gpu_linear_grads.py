"""The two float32 gradients of a linear layer in one kernel (tpq_f32_linear_grads) against float64."""
import pytest
import torch

from tensorplay_amd import ops
from tensorplay_amd.ao import quantization as q

pytestmark = pytest.mark.gpu


def _case(m, k, n, seed=0):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    g = torch.randn(m, n, device="cuda", generator=gen) * 1e-3
    x = torch.randn(m, k, device="cuda", generator=gen)
    w = torch.randn(n, k, device="cuda", generator=gen) * 0.02
    return g, x, w


def _grads(g, x, w, **want):
    with torch.no_grad():
        return ops.linear_grads(g, x, w, **want)


# one value, edges of the 128 x 128 tiles and of the 32 k stages, several slices of k on either product, many more rows than columns;
# 9, 46, 129 and 400 slices of one product (a workgroup's parts of one, 3, 9 and 25 of them, the last ones short or empty), and 12 of one
# that is added without parts
SIZES = [(1, 4, 4), (4, 4, 260), (5, 132, 260), (31, 128, 124), (33, 1280, 712), (128, 512, 512), (129, 260, 132), (72, 1280, 4096), (295, 808, 3840), (2100, 96, 64),
         (1150, 64, 68), (129, 1040, 2304), (40, 68, 7300), (16500, 60, 124), (64000, 4, 8)]


@pytest.mark.parametrize("m,k,n", SIZES)
def test_against_float64(m, k, n):
    g, x, w = _case(m, k, n)
    gx, gw = _grads(g, x, w)
    for got, a, b in ((gx, g, w), (gw, g.T, x)):
        want, size = a.double() @ b.double(), a.double().abs() @ b.double().abs()
        # six part products leave out 3 x 2^-24 of a term at most; the chain of float32 sums rounds each of its at most 6 K / 16 steps once
        # (slices only shorten it): 2^-24 of the sum so far, taken as the sum of the magnitudes, with the steps' roundings in all
        # directions (their square root, four times over)
        steps = 6 * ((a.shape[1] + 15) // 16) + 8
        bound = size * (3 * 2.0 ** -24 + 4 * steps ** 0.5 * 2.0 ** -24)
        assert bool(((got.double() - want).abs() <= bound).all())
    torch_err = ((g.T @ x).double() - g.T.double() @ x.double()).norm()
    assert (gw.double() - g.T.double() @ x.double()).norm() <= 1.05 * torch_err + 1e-30  # as exact as the float32 product it replaces


def test_wide_range_of_values_keeps_float32_precision():
    """Rows whose values span 2^60: every term keeps its own 24 bits, nothing is scaled by the largest."""
    g, x, w = _case(64, 256, 256)
    g = g * torch.exp2(torch.randint(-30, 30, (1, 256), device="cuda").float())
    w = w * torch.exp2(torch.randint(-30, 30, (256, 1), device="cuda").float())
    w[g.abs().amax(0) > 1e3] = 0.0  # the largest values meet zeros
    gx, _ = _grads(g, x, w, want_weight=False)
    size = g.double().abs() @ w.double().abs()
    assert bool(((gx.double() - g.double() @ w.double()).abs() <= size * 2.0 ** -20).all())


@pytest.mark.parametrize("power", [-104, -111, -118, -126, -134, -146])
def test_tiny_values_keep_float32_precision(power):
    """Values whose bfloat16 parts are subnormal, or nothing, in a few columns (the second stage of k and the last) and in all, against
    partners of 2^100: the products are ordinary numbers."""
    g, x, w = _case(40, 132, 260)
    tiny = torch.randint(1 << 23, 1 << 24, g.shape, device="cuda").double() * 2.0 ** (power - 23)
    for columns in (slice(40, 41), slice(257, 260), slice(None)):
        a, b = g.clone(), w.clone()
        a[:, columns] = tiny.float()[:, columns]
        b[columns] *= 2.0 ** 100
        a[:, 80:] *= (a[:, 80:].abs() < 1e-30).float()  # (columns of ordinary size would hide what the tiny ones add)
        gx, gw = _grads(a, x, b)
        for got, left, right in ((gx, a, b), (gw, a.T, x)):
            want, size = left.double() @ right.double(), left.double().abs() @ right.double().abs()
            terms = left.shape[1]
            # a chain of float32 sums, its roundings in all directions, and float32's own smallest step for products below its range
            bound = size * (3 * 2.0 ** -24 + 4 * terms ** 0.5 * 2.0 ** -24) + terms * 2.0 ** -149
            assert bool(((got.double() - want).abs() <= bound).all())


@pytest.mark.parametrize("value", [1.1e-39, float("inf")])
def test_one_such_value_changes_its_own_tiles_only(value):
    """Several tiles of rows and columns and slices of k in both products, the value in a tile and a slice in the middle."""
    g, x, w = _case(650, 520, 1100)
    before = _grads(g, x, w)
    g[300, 500] = value
    gx, gw = _grads(g, x, w)
    rows = torch.ones(650, dtype=torch.bool, device="cuda")
    rows[256:384] = False  # grad_x: the tile of row 300
    channels = torch.ones(1100, dtype=torch.bool, device="cuda")
    channels[384:512] = False  # grad_w: the tile of channel 500
    assert torch.equal(gx[rows], before[0][rows]) and torch.equal(gw[channels], before[1][channels])
    rows[300] = channels[500] = True
    for got, a, b, own, others in ((gx, g, w, 300, ~rows), (gw, g.T, x, 500, ~channels)):
        want, size = a.double() @ b.double(), a.double().abs() @ b.double().abs()
        bound = size * (3 * 2.0 ** -24 + 4 * a.shape[1] ** 0.5 * 2.0 ** -24)
        assert bool(((got.double() - want).abs() <= bound)[others].all())
        if value > 1:
            assert torch.equal(got[own].double(), want[own]) and bool(got[own].isinf().all())
        else:
            assert bool(((got.double() - want).abs() <= bound)[own].all())


@pytest.mark.parametrize("terms", [1, 2, 3, 4])
def test_sums_of_few_terms_round_once_a_term(terms):
    from tensorplay_amd import _lib

    g, x, w = _case(terms, 132, 260)
    gx, gw = torch.empty_like(x), torch.empty_like(w)
    scratch = torch.empty(1 << 22, dtype=torch.uint8, device="cuda")  # the kernel itself: the operator leaves up to three rows to the products
    assert _lib.load().tpq_f32_linear_grads(g.data_ptr(), x.data_ptr(), w.data_ptr(), terms, 132, 260, gx.data_ptr(), gw.data_ptr(), scratch.data_ptr(),
                                            scratch.numel(), torch.cuda.current_stream().cuda_stream) == _lib.TPQ_OK
    want, size = g.double().T @ x.double(), g.double().abs().T @ x.double().abs()
    if terms < 4:  # float32: half a unit for each product and each sum
        assert bool(((gw.double() - want).abs() <= size * terms * 2.0 ** -24).all())
    assert (gw.double() - want).norm() <= 1.02 * ((g.T @ x).double() - want).norm()


def test_products_next_to_the_largest_value():
    """Factors that round up to 2^64 in bfloat16: the product of the rounded ones is infinite, theirs is not."""
    g, x, w = _case(8, 64, 64)
    g[2], w[:, 5] = 0.0, 0.0
    g[2, 7] = w[7, 5] = 2.0 ** 64 * (1 - 2.0 ** -12)
    gx, _ = _grads(g, x, w, want_weight=False)
    want = g.double() @ w.double()
    assert bool(gx.isfinite().all()) and float(gx[2, 5]) == float(want[2, 5].float())
    assert bool(((gx.double() - want).abs() <= 1e-5 * (g.double().abs() @ w.double().abs())).all())


def test_infinities_and_nan_as_in_float32():
    g, x, w = _case(40, 132, 260)
    g[3, 7], g[4, 8], g[5, 9], g[6, 1] = float("inf"), float("-inf"), float("nan"), 3.4e38
    w[8] = 0.0  # -inf x 0
    w[1] = 1.0
    gx, gw = _grads(g, x, w)
    for got, want in ((gx, g.cpu().double() @ w.cpu().double()), (gw, g.cpu().double().T @ x.cpu().double())):
        want = want.float().cpu()
        got = got.cpu()
        assert torch.equal(got.isnan(), want.isnan())
        assert torch.equal(got.isposinf(), want.isposinf()) and torch.equal(got.isneginf(), want.isneginf())


def test_one_gradient_and_leading_dims():
    g, x, w = _case(24, 64, 128)
    gx, gw = _grads(g.view(2, 3, 4, 128), x.view(2, 3, 4, 64), w)
    only_x, none = _grads(g, x, w, want_weight=False)
    nothing, only_w = _grads(g, x, w, want_input=False)
    assert none is None and nothing is None and gx.shape == (2, 3, 4, 64)
    assert torch.equal(gx.view(24, 64), only_x) and torch.allclose(gw, only_w, rtol=1e-5, atol=1e-9)


def test_forms_that_stay_with_the_plain_products():
    """Sizes that are no multiple of 4, other layouts and types, an address off 16 bytes, a recorded backward."""
    for m, k, n in ((5, 6, 8), (5, 8, 6)):
        g, x, w = _case(m, k, n)
        gx, gw = _grads(g, x, w)
        assert torch.allclose(gx, g @ w, rtol=1e-5, atol=1e-8) and torch.allclose(gw, g.T @ x, rtol=1e-5, atol=1e-8)
    g, x, w = _case(16, 64, 32)
    for other in (g.T.contiguous().T, torch.randn(16 * 32 + 1, device="cuda")[1:].view(16, 32), g[:1].expand(16, 32)):
        gx, gw = _grads(other, x, w)
        assert torch.allclose(gx, other @ w, rtol=1e-5, atol=1e-6) and torch.allclose(gw, other.T @ x, rtol=1e-5, atol=1e-5)
    lin = q.Int8DynActInt4WeightLinear(64, 32, bias=False, device="cuda")
    x = x.requires_grad_()
    grad = g.clone().requires_grad_()
    gx, = torch.autograd.grad(lin(x), x, grad, create_graph=True)
    second, = torch.autograd.grad(gx.square().sum(), grad)
    assert torch.allclose(second, 2 * (g @ lin.weight) @ lin.weight.T, rtol=1e-4, atol=1e-7)


@pytest.mark.parametrize("frozen", [False, True])
def test_a_16_bit_layer_refuses_its_backward(frozen):
    """Its output and the gradient of that are float32: no product with 16-bit operands, with the weight's gradient wanted or not."""
    lin = q.Int8DynActInt4WeightLinear(64, 32, bias=False, device="cuda").bfloat16()
    lin.weight.requires_grad_(not frozen)
    x = torch.randn(16, 64, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    with pytest.raises(RuntimeError):
        lin(x).sum().backward()


def test_tangents_pass_through_the_backward():
    """The derivative of the gradients along a direction of the output's gradient, in forward mode."""
    import torch.autograd.forward_ad as fwad

    lin = q.Int8DynActInt4WeightLinear(64, 32, bias=False, device="cuda")
    g, x, _ = _case(16, 64, 32)
    along = torch.randn_like(g)
    x = x.requires_grad_()
    out = lin(x)
    with fwad.dual_level():
        gx, gw = torch.autograd.grad(out, (x, lin.weight), fwad.make_dual(g, along))
        gx, gw = fwad.unpack_dual(gx), fwad.unpack_dual(gw)
    for got, want in ((gx.tangent, along @ lin.weight), (gw.tangent, along.T @ x), (gx.primal, g @ lin.weight), (gw.primal, g.T @ x)):
        assert got is not None and torch.allclose(got, want, rtol=1e-4, atol=1e-6)


def test_module_gradients_replay_in_a_graph():
    lin = q.Int8DynActInt4WeightLinear(512, 768, bias=False, device="cuda")
    x = torch.randn(96, 512, device="cuda", requires_grad=True)
    grad = torch.randn(96, 768, device="cuda")
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        torch.autograd.grad(lin(x), (x, lin.weight), grad)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = torch.autograd.grad(lin(x), (x, lin.weight), grad)
    for seed in range(3):
        with torch.no_grad():
            grad.copy_(torch.randn(96, 768, device="cuda", generator=torch.Generator(device="cuda").manual_seed(seed)))
        graph.replay()
        torch.cuda.synchronize()
        eager = torch.autograd.grad(lin(x), (x, lin.weight), grad)
        assert all(torch.equal(a, b) for a, b in zip(out, eager))
