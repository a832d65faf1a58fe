"""GPU: packed weights against a block of activation rows (tpq_int4_mm_rows, tpq_lowbit_mm_rows), every element within the
bound that its roundings give, against float64 on the same quantized operands."""
import ctypes

import numpy as np
import pytest
import torch

from gpu_util import DEV

pytestmark = pytest.mark.gpu

STAGED, QUADS_OF_ROWS, LANES_OF_CHANNELS = 0, 1, 2  # the kernels: activations staged in LDS; float32 in blocks of four rows, with a lane per channel


def _plan(dtype, M, N, K, bits, group, room=-1):
    """[kernel, rows of a tile, its channels, slices of k] of a call with a workspace of `room` bytes (-1: what it asks for); bits 0: the int4 layout."""
    from tensorplay_amd import _lib, ops

    out = (ctypes.c_int32 * 4)()
    ops._check(_lib.load().tpq_packed_rows_call_plan(ops._DT[dtype], M, N, K, bits, group, room, ctypes.cast(out, ctypes.c_void_p)))
    return list(out)


UNIT = {torch.float32: 2.0 ** -24, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}
# (M, N, K, group): one and two rounds of four steps of 128 k, rounds of which the last is partial, several slices of k, rows at
# and one past the edges of 16- and 64-row tiles, channels that leave a tile of 64 (128) partly empty, a last step of 32, 64, 96 k
SHAPES = [(1, 64, 32, 32), (16, 72, 512, 128), (17, 136, 544, 32), (33, 264, 1024, 64), (48, 64, 2048, 128), (49, 200, 4032, 64),
          (64, 520, 4096, 128), (65, 72, 1152, 128), (128, 1032, 8192, 128), (130, 4104, 608, 32), (200, 2056, 1280, 128),
          # tiles of 80, 96, 112 and 128 rows (16-bit; taken where fewer tall tiles fit the compute units at once), one to four rounds
          (75, 25608, 256, 64), (90, 25608, 640, 128), (112, 25608, 256, 32), (127, 25608, 896, 128)]


def _check(got, x, w, bias, scale_max, dtype):
    x64, w64 = x.double().cpu(), w.double().cpu()
    exact = x64 @ w64.t()
    if bias is not None:
        exact = exact + bias.double().cpu()
    size = x64.abs() @ w64.abs().t()
    u, k = UNIT[dtype], x.shape[1]
    # weights rounded once (not in float32), fp32 sums of k terms, the fp16 offset of a code (at most 1024 + 128) leaving
    # through an fp32 constant of the size of offset x scale, the result rounded once
    bound = ((0 if dtype == torch.float32 else u) + (k + 16) * 2.0 ** -24) * size + u * exact.abs()
    bound = bound + 2 * 1160 * 2.0 ** -24 * scale_max * x64.abs().sum(1, keepdim=True) * (0 if dtype == torch.float32 else 1) + 1e-30
    err = (got.double().cpu() - exact).abs()
    assert torch.isfinite(got).all() and bool((err <= bound).all()), f"{float((err / bound).max()):.3f} times the bound"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,N,K,group", SHAPES)
def test_int4_rows(dtype, M, N, K, group):
    from tensorplay_amd import _lib, ops

    gen = torch.Generator(device=DEV).manual_seed(M + N + K)
    codes = torch.randint(0, 16, (N, K), dtype=torch.int32, device=DEV, generator=gen)
    packed = ops._convert_weight_to_int4pack(codes, 2)
    sz = torch.stack([torch.rand(K // group, N, device=DEV, generator=gen) * 0.01 + 1e-3,
                      torch.randn(K // group, N, device=DEV, generator=gen) * 0.01], -1).to(dtype).contiguous()
    x = torch.randn(M, K, device=DEV, generator=gen).to(dtype)
    w = (codes - 8).double() * sz[..., 0].double().t().repeat_interleave(group, 1) + sz[..., 1].double().t().repeat_interleave(group, 1)
    lib = _lib.load()
    need = int(lib.tpq_packed_rows_call_workspace_bytes(ops._DT[dtype], M, N, K, 0, group))
    for room in {need, 0}:  # with its slices, and without a workspace
        out = torch.empty(M, N, dtype=dtype, device=DEV)
        ws = torch.empty(max(room, 1), dtype=torch.uint8, device=DEV)
        ops._check(lib.tpq_int4_mm_rows(x.data_ptr(), ops._DT[dtype], M, K, packed.data_ptr(), N, group, sz.data_ptr(), out.data_ptr(),
                                        ws.data_ptr() if room else None, room, ops._stream(x)))
        _check(out, x, w, None, 0.011, dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("bits,lsb_first", [(1, False), (1, True), (2, False), (4, False), (8, False)])
@pytest.mark.parametrize("M,N,K,group", [(17, 68, 160, 32), (33, 264, 1056, 96), (64, 200, 4096, 512), (130, 1028, 640, 128), (90, 25604, 256, 32), (127, 25604, 640, 128)])
def test_lowbit_rows(dtype, bits, lsb_first, M, N, K, group):
    from tensorplay_amd import _lib, ops

    gen = torch.Generator(device=DEV).manual_seed(M + N + K + bits)
    codes = torch.randint(0, 1 << bits, (N, K), dtype=torch.uint8, device=DEV, generator=gen)
    packed = ops.pack_lowbit(codes, bits, lsb_first)
    sz = torch.stack([torch.rand(K // group, N, device=DEV, generator=gen) * 0.01 + 1e-3,
                      torch.rand(K // group, N, device=DEV, generator=gen) * (1 << bits)], -1).contiguous()
    bias = torch.randn(N, device=DEV, generator=gen)
    x = torch.randn(M, K, device=DEV, generator=gen).to(dtype)
    value = (codes.view(torch.int8) if bits == 8 else codes).double()  # 8-bit codes are signed
    scale, zero = (sz[..., i].double().t().repeat_interleave(group, 1) for i in (0, 1))
    w = (value - zero) * scale
    out = torch.empty(M, N, dtype=dtype, device=DEV)
    lib = _lib.load()
    need = int(lib.tpq_packed_rows_call_workspace_bytes(ops._DT[dtype], M, N, K, bits, group))
    assert need > 0 or (M, N, K) not in ((33, 264, 1056), (64, 200, 4096))  # slices with a last step that is partial, and many
    ws = torch.empty(max(need, 1), dtype=torch.uint8, device=DEV)
    ops._check(lib.tpq_lowbit_mm_rows(x.data_ptr(), ops._DT[dtype], M, K, packed.data_ptr(), bits, int(lsb_first), N, group, sz.data_ptr(),
                                      bias.data_ptr(), out.data_ptr(), ws.data_ptr(), need, ops._stream(x)))
    # the zero point and the code meet after their products with the scale: |zero| scale on top of |w|
    _check(out, x, w, bias, 0.011 * (1 + (1 << bits) / 8), dtype)


# (M, N, K, group, (rows of a tile, slices of k) for int4, 1 to 4 and 8 bits): two to four tiles of rows, the last one partly empty, whole k and cut
TALL = [(257, 6664, 256, 64, (80, 1), (80, 1), (80, 1)), (241, 8200, 256, 32, (96, 1), (96, 1), (96, 1)), (289, 8200, 256, 128, (112, 1), (112, 1), (112, 1)),
        (225, 11016, 256, 64, (128, 1), (128, 1), (128, 1)), (257, 1096, 5248, 128, (80, 7), (80, 7), (80, 7)), (241, 1544, 7296, 64, (96, 6), (96, 6), (64, 2)),
        (289, 1608, 7296, 128, (112, 6), (80, 4), (80, 4)), (241, 2824, 7296, 128, (128, 5), (64, 1), (128, 5)), (203, 11008, 4096, 128, (112, 1), (112, 1), (112, 1)),
        (193, 4104, 3840, 128, (48, 1), (48, 1), (112, 3)), (257, 2056, 7296, 128, (96, 5), (96, 5), (96, 5))]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bits", [0, 1, 2, 8])  # 0: the int4 layout
@pytest.mark.parametrize("M,N,K,group,int4,few_bits,byte", TALL)
def test_tall_tiles(dtype, bits, M, N, K, group, int4, few_bits, byte):
    kernel, rows, _, slices = _plan(dtype, M, N, K, bits, group)
    assert kernel == STAGED and (rows, slices) == {0: int4, 8: byte}.get(bits, few_bits)
    if bits:
        test_lowbit_rows(dtype, bits, False, M, N, K, group)
    else:
        test_int4_rows(dtype, M, N, K, group)


def _fragment(kind, M, N, K, group, bits, dtype, change=lambda x, sz: None):
    """(result, exact float64 result) on weights whose (scale, zero) have no short form in 16 bits.  change: of x and the pairs, in
    place, before the call (sz [K / group, N, 2], of the type that the call takes)."""
    from tensorplay_amd import ops

    gen = torch.Generator(device=DEV).manual_seed(M + N + K + bits)
    x = torch.randn(M, K, device=DEV, generator=gen).to(dtype)
    sz = torch.rand(K // group, N, 2, device=DEV, generator=gen) * 0.01 + 0.001
    if kind == "int4":
        codes = torch.randint(0, 16, (N, K), dtype=torch.int32, device=DEV, generator=gen)
        packed, sz = ops._convert_weight_to_int4pack(codes, 2), sz.to(dtype)
        change(x, sz)
        w = (codes.double() - 8).view(N, -1, group) * sz[..., 0].double().t()[..., None] + sz[..., 1].double().t()[..., None]
        got = ops._weight_int4pack_mm(x, packed, group, sz)
    else:
        sz[..., 1] *= 100
        change(x, sz)
        per_byte = 8 // bits
        packed = torch.randint(0, 256, (N, K // per_byte), dtype=torch.uint8, device=DEV, generator=gen)
        shifts = torch.arange(8 - bits, -1, -bits, device=DEV)
        codes = ((packed.int()[..., None] >> shifts) & ((1 << bits) - 1)).reshape(N, K)
        if bits == 8:
            codes = codes.to(torch.int8)
        w = (codes.double().view(N, -1, group) - sz[..., 1].double().t()[..., None]) * sz[..., 0].double().t()[..., None]
        got = ops._lowbit_mm(x, packed, bits, K, sz)
    return got, x.double().cpu() @ w.view(N, K).cpu().t().contiguous()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("kind,M,N,K,group,bits", [("int4", 3, 72, 544, 32, 4), ("int4", 33, 520, 608, 32, 4), ("int4", 48, 11008, 1024, 128, 4),
                                                   ("intx", 5, 72, 544, 32, 2), ("intx", 33, 264, 1024, 128, 1), ("intx", 40, 200, 4032, 64, 4),
                                                   ("intx", 49, 520, 1024, 128, 8), ("intx", 80, 136, 2048, 32, 4)])
def test_weights_are_not_rounded_where_the_kernels_before_kept_them(dtype, kind, M, N, K, group, bits):
    """The result is the exact sum rounded once.  Per term the weight is off by 2^-18 (bfloat16: two parts of 8 bits) or, beside the
    result's rounding, by nothing (float16), so with sums of random signs at most about one result in 2^9 lands on the other side
    of a rounding boundary; cancellation moves some more.  A weight rounded to the type moves about four in ten."""
    got, exact = _fragment(kind, M, N, K, group, bits, dtype)
    moved = (got.cpu() != exact.to(dtype)).float().mean().item()
    assert moved < 0.05, moved


@pytest.mark.parametrize("bits", [1, 4, 8])
def test_float32_sums_are_not_one_chain(bits):
    """A rounding is off by 0.41 x 2^-24 of the partial sum (root mean square); chains of 16, 8 and 8 terms whose partial sums grow
    like a random walk give 0.41 x 2^-24 sqrt(32 / 2) = 1e-7 of the result, the offset and the parts' sums a little more; one chain
    of 1024 terms gives five times that."""
    got, exact = _fragment("intx", 19, 4096, 4096, 128, bits, torch.float32)
    assert ((got.cpu().double() - exact).norm() / exact.norm()).item() < 2e-7


# (kind, M, N, K, group, bits): where a 16-bit weight's remainder is multiplied too; a last step that is partial, whole steps, slices of k
SPLIT_SHAPES = [("int4", 5, 72, 544, 32, 4), ("int4", 48, 11008, 1024, 128, 4), ("intx", 33, 264, 1056, 32, 2), ("intx", 40, 72, 8192, 128, 4),
                ("intx", 35, 72, 1024, 128, 8)]


def _assert_same_classes(got, exact):
    """NaN, +inf and -inf where the exact sums are, anything finite elsewhere."""
    got = got.double().cpu()
    assert torch.equal(got.isnan(), exact.isnan())
    assert torch.equal(got.isposinf(), exact.isposinf()) and torch.equal(got.isneginf(), exact.isneginf())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("kind,M,N,K,group,bits", SPLIT_SHAPES)
def test_non_finite_activations(dtype, kind, M, N, K, group, bits):
    """An infinite activation gives +-inf with the sign of its product, NaN only where infinities of both signs or a NaN meet."""
    def change(x, sz):
        x[0, 5], x[1, K - 1], x[2, 3], x[2, K // 2] = float("inf"), float("-inf"), float("inf"), float("inf")
        if M > 4:
            x[4, K - 2], x[M - 1, 40] = float("nan"), float("inf")

    got, exact = _fragment(kind, M, N, K, group, bits, dtype, change)
    _assert_same_classes(got, exact)
    fine = exact.isfinite()
    assert ((got.double().cpu() - exact)[fine].norm() / exact[fine].norm()).item() < max(UNIT[dtype], 3e-7)  # float32: as the sums of ordinary operands


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_infinite_weights_beside_a_partial_step(dtype):
    """A zero point that is infinite in the last group of a K that ends inside a step: positive activations give +inf."""
    def change(x, sz):
        x.abs_().add_(0.1)
        sz[-1, 7, 1] = float("inf")

    got, exact = _fragment("int4", 19, 72, 544, 32, 4, dtype, change)
    assert bool(exact[:, 7].isposinf().all())
    _assert_same_classes(got, exact)


@pytest.mark.parametrize("kind,M,N,K,group,bits", SPLIT_SHAPES)
def test_weights_beyond_float16(kind, M, N, K, group, bits):
    """Weights of 10^5, beyond float16, with activations that bring the sums back into its range."""
    def change(x, sz):
        sz[..., 0] *= 2.0 ** (16 if bits == 8 else 21 if kind == "int4" else 23)
        if kind == "int4":
            sz[..., 1] *= 2.0 ** 21
        x *= 2.0 ** -14

    got, exact = _fragment(kind, M, N, K, group, bits, torch.float16, change)
    assert bool(got.isfinite().all())
    assert ((got.double().cpu() - exact).norm() / exact.norm()).item() < UNIT[torch.float16]


@pytest.mark.parametrize("first", [0, -14, 8])
@pytest.mark.parametrize("power", [0, -10, -16])
@pytest.mark.parametrize("kind,M,N,K,group,bits", SPLIT_SHAPES)
def test_float16_weights_of_any_size_are_not_rounded(kind, M, N, K, group, bits, power, first):
    """(scale, zero) 2^power times the ordinary ones, those of a channel's first group 2^first times the others (where that is the
    larger one, its activations are zero, so that the others count): the exact sum rounded once, as with ordinary weights."""
    def change(x, sz):
        factor = torch.full((K // group, 1), 2.0 ** (max(power, -10) if kind == "int4" else power), device=DEV)
        factor[0] *= 2.0 ** first
        sz[..., 0] *= factor
        if kind == "int4":
            sz[..., 1] *= factor
        x *= 2.0 ** min(-power, 12)
        if first > 0:
            x[:, :group] = 0.0

    got, exact = _fragment(kind, M, N, K, group, bits, torch.float16, change)
    assert bool((exact.abs() > 2.0 ** -14).float().mean() > 0.9)  # the result's own rounding is a normal one
    moved = (got.cpu() != exact.to(torch.float16)).float().mean().item()
    assert moved < 0.05, moved


# (rows, N, K, group): few rows on 32 channels a workgroup and eight steps of k a round: one, two and four rounds, the last one and the last
# step partial, channels that leave a tile partly empty, one tile and more than the compute units
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,N,K,group", [(1, 8, 1024, 32), (16, 40, 1152, 64), (5, 1160, 1376, 32), (32, 72, 2048, 64), (17, 8168, 928, 32), (17, 8200, 928, 32), (29, 2056, 4096, 64)])
def test_few_rows_without_slices(dtype, M, N, K, group):
    from tensorplay_amd import _lib, ops

    if dtype == torch.float32 and M > 16:
        pytest.skip("two blocks of float32 rows do not fit a round of eight steps")
    for bits in (0, 2):
        kernel, rows, channels, slices = _plan(dtype, M, N, K, bits, group, 0)
        if dtype == torch.float32 and M <= 8:
            assert kernel == QUADS_OF_ROWS
        else:  # (8200 channels are a tile of 32 more than there are compute units)
            assert (kernel, rows, channels, slices) == (STAGED, -(-M // 16) * 16, 64 if N == 8200 else 32, 1)
    lib, tag = _lib.load(), ops._DT[dtype]
    gen = torch.Generator(device=DEV).manual_seed(M + N + K)
    x = torch.randn(M, K, device=DEV, generator=gen).to(dtype)
    codes = torch.randint(0, 16, (N, K), dtype=torch.int32, device=DEV, generator=gen)
    sz = torch.stack([torch.rand(K // group, N, device=DEV, generator=gen) * 0.01 + 1e-3, torch.randn(K // group, N, device=DEV, generator=gen) * 0.01], -1).to(dtype).contiguous()
    packed = ops._convert_weight_to_int4pack(codes, 2)
    w = (codes - 8).double() * sz[..., 0].double().t().repeat_interleave(group, 1) + sz[..., 1].double().t().repeat_interleave(group, 1)
    out = torch.empty(M, N, dtype=dtype, device=DEV)
    ops._check(lib.tpq_int4_mm_rows(x.data_ptr(), tag, M, K, packed.data_ptr(), N, group, sz.data_ptr(), out.data_ptr(), None, 0, ops._stream(x)))
    _check(out, x, w, None, 0.011, dtype)
    sz = torch.stack([torch.rand(K // group, N, device=DEV, generator=gen) * 0.01 + 1e-3, torch.randint(0, 4, (K // group, N), device=DEV, generator=gen).float()], -1).contiguous()
    codes = torch.randint(0, 4, (N, K), dtype=torch.int32, device=DEV, generator=gen)
    packed = ((codes.view(N, K // 4, 4) << torch.tensor([6, 4, 2, 0], device=DEV, dtype=torch.int32)).sum(-1)).to(torch.uint8).contiguous()
    w = (codes.double() - sz[..., 1].double().t().repeat_interleave(group, 1)) * sz[..., 0].double().t().repeat_interleave(group, 1)
    ops._check(lib.tpq_lowbit_mm_rows(x.data_ptr(), tag, M, K, packed.data_ptr(), 2, 0, N, group, sz.data_ptr(), None, out.data_ptr(), None, 0, ops._stream(x)))
    _check(out, x, w, None, 0.011, dtype)


def test_few_rows_take_no_workspace():
    """The plan's side of it: no slices where a few thousand k go to 32 channels a workgroup, slices beyond."""
    from tensorplay_amd import _lib, ops

    lib, f16 = _lib.load(), ops._DT[torch.float16]
    assert lib.tpq_packed_rows_workspace_bytes(f16, 28, 4096, 4096) == 0 and lib.tpq_packed_rows_workspace_bytes(f16, 20, 2048, 2048) == 0
    assert lib.tpq_packed_rows_workspace_bytes(f16, 33, 2048, 2048) > 0 and lib.tpq_packed_rows_workspace_bytes(f16, 28, 4096, 11008) > 0
    assert lib.tpq_lowbit_mm_rows_workspace_bytes(f16, 3, 5832, 2944) == 0


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K,group", [(46, 1688, 1824, 32), (2, 3032, 4640, 32), (11, 1184, 3136, 64), (33, 1024, 4096, 128)])
def test_calls_have_the_slices_that_their_weight_wants(dtype, M, N, K, group):
    """A weight that is not rounded (K % 128 != 0, groups of 128 on few rows) has longer rounds of the loop than one that is, and slices where
    that has none: the Python entry gives the library room for them (one slice adds k in another order: some outputs in a thousand differ)."""
    from tensorplay_amd import _lib, ops

    lib, tag = _lib.load(), ops._DT[dtype]
    need = int(lib.tpq_packed_rows_call_workspace_bytes(tag, M, N, K, 0, group))
    slices = _plan(dtype, M, N, K, 0, group, need)[3]
    assert need == 4 * slices * M * N and slices > 1
    gen = torch.Generator(device=DEV).manual_seed(M + N + K)
    packed = ops._convert_weight_to_int4pack(torch.randint(0, 16, (N, K), dtype=torch.int32, device=DEV, generator=gen), 2)
    sz = (torch.rand(K // group, N, 2, device=DEV, generator=gen) * 0.01 + 1e-3).to(dtype)
    x = torch.randn(M, K, device=DEV, generator=gen).to(dtype)
    assert lib.tpq_int4_mm_rows_takes(x.data_ptr(), tag, M, N, K, group, packed.data_ptr(), sz.data_ptr())
    results = []
    for room in (need, 0):
        out, ws = torch.empty(M, N, dtype=dtype, device=DEV), torch.empty(max(room, 16), dtype=torch.uint8, device=DEV)
        ops._check(lib.tpq_int4_mm_rows(x.data_ptr(), tag, M, K, packed.data_ptr(), N, group, sz.data_ptr(), out.data_ptr(), ws.data_ptr() if room else None, room, ops._stream(x)))
        results.append(out)
    assert not torch.equal(*results)
    assert torch.equal(ops._weight_int4pack_mm(x, packed, group, sz), results[0])


# (M, N, K, group): float32 in blocks of four rows: one and two blocks, full and not; steps of 128 k of which the last one has one to three tiles, fewer
# steps than wavefronts, more than they have in flight; a part of 32 and of 64 channels; slices of k
QUADS = [(1, 4, 32, 32), (3, 40, 96, 96), (4, 32, 160, 32), (5, 68, 1088, 64), (8, 200, 4096, 128), (4, 1160, 8224, 32), (7, 9736, 4864, 128), (2, 8200, 3072, 64)]


def _float32_products(counts, N, K, group, bits, lsb_first):
    """The first rows of one x, as many as each count says, with a bias, with the plan's slices and without a workspace, every element within its bound of float64: ({count: result}, |x| |w|)."""
    from tensorplay_amd import _lib, ops

    lib, tag, most = _lib.load(), ops._DT[torch.float32], max(counts)
    gen = torch.Generator(device=DEV).manual_seed(most + N + K + bits)
    x = torch.randn(most, K, device=DEV, generator=gen)
    bias = torch.randn(N, device=DEV, generator=gen)
    codes = torch.randint(0, 1 << (bits or 4), (N, K), dtype=torch.int32, device=DEV, generator=gen)
    scale, zero = torch.rand(K // group, N, device=DEV, generator=gen) * 0.01 + 1e-3, torch.randn(K // group, N, device=DEV, generator=gen)
    sz = torch.stack([scale, zero * (1.0 if bits else 0.01)], -1).contiguous()
    s64, z64 = (sz[..., i].double().t().repeat_interleave(group, 1) for i in (0, 1))
    if bits == 0:
        packed = ops._convert_weight_to_int4pack(codes, 2)
        w = (codes - 8).double() * s64 + z64
    else:
        codes = codes - 128 if bits == 8 else codes
        per = 8 // bits
        order = [i * bits if lsb_first else 8 - (i + 1) * bits for i in range(per)]
        packed = ((codes & 255).view(N, K // per, per) << torch.tensor(order, device=DEV, dtype=torch.int32)).sum(-1).to(torch.uint8).contiguous()
        w = (codes.double() - z64) * s64
    results = {}
    for m in counts:
        sizes = {int(lib.tpq_packed_rows_call_workspace_bytes(tag, m, N, K, bits, group)), 0}
        for need in sizes:
            out = torch.full((m, N), float("nan"), device=DEV)
            ws = torch.empty(max(need, 1), dtype=torch.uint8, device=DEV)
            at = [x.data_ptr(), tag, m, K, packed.data_ptr()], [bias.data_ptr(), out.data_ptr(), ws.data_ptr() if need else None, need, ops._stream(x)]
            if bits:
                ops._check(lib.tpq_lowbit_mm_rows(*at[0], bits, int(lsb_first), N, group, sz.data_ptr(), *at[1]))
            else:
                ops._check(lib.tpq_int4_mm_rows_bias(*at[0], N, group, sz.data_ptr(), *at[1]))
            _check(out, x[:m], w, bias, 0.011, torch.float32)
            results[m] = out
    return results, x.double().abs() @ w.abs().t() + bias.double().abs()


WIDTHS = [(0, False), (1, False), (1, True), (2, False), (4, False), (8, False)]  # (bits, lsb_first), 0: the int4 layout


@pytest.mark.parametrize("bits,lsb_first", WIDTHS)
@pytest.mark.parametrize("M,N,K,group", QUADS)
def test_blocks_of_four_rows(M, N, K, group, bits, lsb_first):
    """Against float64, element by element, and beside the kernels of 16 rows: the same rows among nine, whose bound is the same."""
    N, group = (N + 7) // 8 * 8 if bits == 0 else N, group if bits or group in (32, 64, 128) else 32
    assert _plan(torch.float32, M, N, K, bits, group)[:2] == [QUADS_OF_ROWS, 4 * -(-M // 4)] and _plan(torch.float32, 9, N, K, bits, group)[0] != QUADS_OF_ROWS
    results, size = _float32_products((M, 9), N, K, group, bits, lsb_first)
    assert bool(((results[M] - results[9][:M]).double().abs() <= 2 * (K + 17) * 2.0 ** -24 * size[:M]).all())


# (M, N, K, group, rows of a tile, widths whose plan it is): float32 with a lane per channel: one to four blocks of 16 rows, with a block of four behind one to three of
# them, full and not, two and three tiles of rows; fewer tiles of k than wavefronts, more than they have in flight; channels that leave a part partly empty
ALL, INT4, BITS, BYTE = (0, 1, 2, 4, 8), (0,), (1, 2, 4), (8,)
LANES = [(17, 8200, 96, 32, 20, ALL), (20, 8200, 1088, 32, 20, ALL), (17, 68, 11008, 128, 20, ALL), (35, 1032, 4128, 32, 36, ALL), (52, 1032, 2080, 32, 52, INT4 + BYTE),
         (14, 11008, 4096, 128, 16, INT4), (40, 4096, 4096, 128, 48, ALL), (60, 4096, 4096, 64, 64, INT4 + BITS), (96, 2056, 2080, 32, 48, ALL), (130, 1032, 4096, 64, 48, INT4 + BITS),
         (14, 68, 1088, 32, 16, BITS + BYTE), (29, 68, 544, 32, 32, ALL), (50, 68, 544, 32, 52, ALL), (60, 68, 544, 32, 64, ALL)]


@pytest.mark.parametrize("M,N,K,group,rows,bits,lsb_first", [(*shape, bits, lsb_first) for *shape, widths in LANES for bits, lsb_first in WIDTHS if bits in widths])
def test_lane_per_channel(M, N, K, group, rows, bits, lsb_first):
    """Against float64, element by element, and beside the blocks of four: the first eight rows by themselves."""
    N = (N + 7) // 8 * 8 if bits == 0 else N
    assert _plan(torch.float32, M, N, K, bits, group)[:2] == [LANES_OF_CHANNELS, rows]
    results, size = _float32_products((M, 8), N, K, group, bits, lsb_first)
    assert bool(((results[M][:8] - results[8]).double().abs() <= 2 * (K + 17) * 2.0 ** -24 * size[:8]).all())


# (M, N, K, group, bits): wide layers over a long k, whose plan cuts it little or not at all, at every height of a tile with a lane per channel
LONG = [(16, 3712, 9984, 128, 0), (13, 13440, 1792, 32, 0), (19, 11008, 4096, 128, 0), (32, 9728, 4096, 128, 2), (36, 8192, 5632, 64, 4), (48, 8192, 4096, 128, 1), (66, 7552, 2944, 128, 4),
        (35, 4736, 6272, 128, 8), (141, 3712, 5888, 32, 0)]


@pytest.mark.parametrize("M,N,K,group,bits", LONG)
def test_float32_sums_keep_the_precision_of_steps(M, N, K, group, bits):
    """The error against float64 is no larger than that of sums over 16 k, eight of those over a step of 128 and a quarter of the steps in a chain (on 192 channels; 3 % for
    what two samples of 2500 to 27 000 outputs differ by): one chain of the sums of 16 k over a long slice has up to a fifth more."""
    from tensorplay_amd import ops

    gen = torch.Generator(device=DEV).manual_seed(M + N + K + bits)
    x = torch.randn(M, K, device=DEV, generator=gen)
    w = torch.randn(N, K, device=DEV, generator=gen).mul_(0.02).view(N, K // group, group)
    lo, hi = w.amin(-1), w.amax(-1)
    least, levels = (-128 if bits == 8 else -8 if bits == 0 else 0), (1 << (bits or 4)) - 1
    scale = (hi - lo) / levels
    zero = least - lo / scale if bits == 0 else (least - lo / scale).round()
    codes = ((w / scale[..., None]) + zero[..., None]).round_().clamp_(least, least + levels).int()
    if bits == 0:
        sz = torch.stack([scale.t(), (-zero * scale).t()], -1).contiguous()
        got = ops._weight_int4pack_mm(x, ops._convert_weight_to_int4pack((codes + 8).view(N, K), 2), group, sz)
    else:
        sz = torch.stack([scale.t(), zero.t()], -1).contiguous()
        got = ops._lowbit_mm(x, ops.pack_lowbit((codes.view(N, K) & 255).to(torch.uint8), bits, False), bits, K, sz)
    rows = slice(0, 192)
    s64, z64 = sz[..., 0].t()[rows, :, None].double(), sz[..., 1].t()[rows, :, None].double()
    c64 = codes[rows].double()
    exact_w = (c64 * s64 + z64 if bits == 0 else (c64 - z64) * s64).view(192, K)
    exact = x.double() @ exact_w.t()
    pieces = torch.stack([x[:, k : k + 16] @ exact_w.float()[:, k : k + 16].t() for k in range(0, K, 16)], -1)
    pieces = torch.nn.functional.pad(pieces, (0, -pieces.shape[-1] % 32))

    def chain(t):
        total = t[..., 0].clone()
        for i in range(1, t.shape[-1]):
            total += t[..., i]
        return total

    steps = chain(pieces.view(M, 192, -1, 8))
    quarters = chain(steps.view(M, 192, -1, 4).transpose(-1, -2))
    reference = (quarters[..., 0] + quarters[..., 1]) + (quarters[..., 2] + quarters[..., 3])

    def error(y):
        return float((y.double() - exact).norm() / exact.norm())

    assert error(got[:, rows]) <= 1.03 * error(reference), (error(got[:, rows]), error(reference))


@pytest.mark.parametrize("kind,bits", [("int4", 4), ("lowbit", 1), ("lowbit", 8)])
@pytest.mark.parametrize("M", [6, 19])  # blocks of four; a lane per channel
def test_float32_rows_not_finite(M, kind, bits):
    """Infinite activations and zero points, in the last tile of a K that ends inside a step of 128."""
    def change(x, sz):
        x[0, 5], x[1, -1], x[2, 3], x[2, 40] = float("inf"), float("-inf"), float("inf"), float("nan")
        sz[-1, 7, 1] = float("inf")

    _assert_same_classes(*_fragment(kind, M, 72, 544, 32, bits, torch.float32, change))
