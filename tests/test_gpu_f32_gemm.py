"""The fp32-activation GEMM over exact bf16 pieces (batches past one decode pass) at the edges of its
tiles: 32- and 64-token tiles, 256-feature workgroups, K splits down to two 64-wide stages, one and two
stages per group, nibble and byte codes, against float64.

Bound per output: the operands and products are exact, so the error is that of the fp32 sums -- at most
3 x group products and the folds of the K / group group sums, each of relative size u = 2^-23 (one ulp,
for any rounding), of the magnitudes |s| (|q - zi| + |z - zi|) |x| that enter them; three pieces of x
sum to at most (1 + 2^-7) |x| in magnitude."""

from __future__ import annotations

import pytest
import torch

from llmopt.kernels import ops
from llmopt.quantization import QuantizedTensor

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _weight(n, k, bits, group, symmetric, seed, zeros="int"):
    g = torch.Generator().manual_seed(seed)
    codes = torch.randint(0, 1 << bits, (n, k), generator=g)
    scales = torch.rand(n, k // group, generator=g) * 0.01 + 0.002
    mid = float(1 << (bits - 1))
    if symmetric:
        points = torch.full_like(scales, mid)
        z = torch.zeros_like(scales)
    else:
        points = torch.randint(0, 1 << bits, scales.shape, generator=g).float()
        if zeros == "fraction":
            points = points + torch.randint(0, 2, scales.shape, generator=g) * 0.375
        elif zeros == "far":
            points = points - 3000.0 * torch.randint(0, 2, scales.shape, generator=g)
        z = points
    if bits == 8:
        q = (codes - 128).to(torch.int8) if symmetric else codes.to(torch.uint8)
    else:
        c = codes.to(torch.uint8)
        q = c[:, 0::2] | (c[:, 1::2] << 4)
    qt = QuantizedTensor(q.contiguous().to(DEV), scales.to(DEV), z.to(DEV), bits, group, symmetric, (n, k))
    d = codes.view(n, -1, group).double() - points.double()[..., None]
    w = (d * scales.double()[..., None]).view(n, k).to(DEV)
    # Magnitudes in the sums: the difference itself, or where the integer part is replaced, both parts.
    mag = ((codes.view(n, -1, group).double() + points.double().abs()[..., None] + mid) *
           scales.double()[..., None]).view(n, k).to(DEV)
    return qt, w, mag if zeros != "int" else w.abs()


def _check(y, x, w, mag, group, bias=None):
    ref = x.double() @ w.t()
    k = x.shape[1]
    bound = (x.double().abs() @ mag.t()) * ((3 * group + k / group + 4) * 2.0**-23 * (1 + 2.0**-7))
    if bias is not None:
        ref = ref + bias.double()
        bound = bound + ref.abs() * 2.0**-23
    assert bool(((y.double() - ref).abs() <= bound + 1e-30).all())


SHAPES = [  # (n, k, bits, group, symmetric): k >= 128, groups of one stage and of several
    (256, 128, 4, 64, True), (257, 256, 4, 128, False), (100, 1152, 4, 64, False), (511, 384, 8, 128, True),
    (320, 1024, 8, 64, False), (513, 512, 2, 256, False), (1024, 4096, 4, 64, True),
]


@pytest.mark.parametrize("shape", range(len(SHAPES)))
@pytest.mark.parametrize("m", [17, 22, 32, 33, 63, 64, 65, 97, 200])
def test_edges_of_tiles(shape, m):
    n, k, bits, group, symmetric = SHAPES[shape]
    qt, w, mag = _weight(n, k, bits, group, symmetric, seed=shape)
    g = torch.Generator().manual_seed(m)
    x = torch.randn(m, k, generator=g).to(DEV)
    bias = torch.randn(n, generator=g).to(DEV) if m % 2 else None
    _check(ops.quant_linear(x, qt, bias, torch.float32), x, w, mag, group, bias)


@pytest.mark.parametrize("zeros", ["fraction", "far"])
@pytest.mark.parametrize("bits,group", [(4, 64), (4, 256), (8, 128)])
def test_zero_points_off_the_integer_range(zeros, bits, group):
    # Zero points that are not integers, or too far for exact bf16 differences: the remainder enters
    # through the sums of x.
    qt, w, mag = _weight(300, 1024, bits, group, False, seed=5, zeros=zeros)
    x = torch.randn(70, 1024, generator=torch.Generator().manual_seed(6)).to(DEV)
    _check(ops.quant_linear(x, qt, None, torch.float32), x, w, mag, group)


def test_unaligned_rows_and_wide_magnitudes():
    n, k, m = 200, 512, 80
    qt, w, mag = _weight(n, k, 4, 64, True, seed=7)
    g = torch.Generator().manual_seed(8)
    base = torch.randn(m, k + 3, generator=g) * torch.exp2(torch.randint(-40, 40, (m, 1), generator=g).float())
    x = base.to(DEV)[:, 1 : k + 1]  # rows off 16-byte alignment, stride k + 3
    _check(ops.quant_linear(x, qt, None, torch.float32), x, w, mag, 64)


def test_infinities_and_nan_match_the_dense_product():
    n, k, m = 64, 256, 40
    qt, w, _ = _weight(n, k, 4, 64, True, seed=9)
    x = torch.randn(m, k, generator=torch.Generator().manual_seed(10)).to(DEV)
    x[3, 17], x[4, 200], x[5, 0] = float("inf"), float("-inf"), float("nan")
    x[6, 9] = 3.0e38  # finite, rounds to infinity in bf16, and overflows times the integer weight
    y = ops.quant_linear(x, qt, None, torch.float32)
    ref = x.double() @ w.t()
    assert torch.equal(torch.isnan(y), torch.isnan(ref))
    assert torch.equal(torch.isposinf(y), torch.isposinf(ref))
    assert torch.equal(torch.isneginf(y), torch.isneginf(ref))
    rest = [0, 1, 2] + list(range(6, m))
    assert bool(((y[rest].double() - ref[rest]).abs() <= 1e-5 * ref[rest].abs().amax(1, keepdim=True)).all())


@pytest.mark.parametrize("zeros", ["fraction", "far"])
@pytest.mark.parametrize("m,n,k,bits,group", [(40, 64, 256, 4, 64), (70, 300, 1024, 4, 128), (65, 257, 768, 8, 64),
                                              (300, 512, 256, 4, 256)])
def test_infinities_with_remainders_of_zero_points(m, n, k, bits, group, zeros):
    # (q - z) x is infinite where (q - zi) x and (z - zi) x have opposite signs or one of them is 0 x: only a
    # weight of exactly zero, or infinities of both signs, make a NaN. Other rows keep their values.
    qt, w, mag = _weight(n, k, bits, group, False, seed=17, zeros=zeros)
    x = torch.randn(m, k, generator=torch.Generator().manual_seed(18)).to(DEV)
    y0 = ops.quant_linear(x, qt, None, torch.float32)
    _check(y0, x, w, mag, group)
    inf = float("inf")
    for row, at in ((3, {17: inf}), (4, {200: -inf}), (5, {0: float("nan")}), (6, {9: inf, 70: inf}),
                    (7, {8: inf, 9: -inf}), (m - 1, {k - 1: inf, 3: 2.0e38})):
        for c, v in at.items():
            x[row, c] = v
    y, ref = ops.quant_linear(x, qt, None, torch.float32), x.double() @ w.t()
    assert torch.equal(torch.isnan(y), torch.isnan(ref))
    assert torch.equal(torch.isposinf(y), torch.isposinf(ref)) and torch.equal(torch.isneginf(y), torch.isneginf(ref))
    rest = [i for i in range(m - 1) if i not in (3, 4, 5, 6, 7)]
    assert torch.equal(y[rest], y0[rest])


@pytest.mark.parametrize("m,n,k,bits,group,symmetric", [(40, 64, 256, 4, 64, True), (70, 300, 1024, 4, 128, False),
                                                        (24, 6144, 4096, 4, 64, True), (65, 200, 768, 8, 768, False),
                                                        (33, 96, 18432, 8, 128, True)])
def test_the_whole_range_of_fp32(m, n, k, bits, group, symmetric):
    # Rows from 2^-140 to the largest finite values, each within the error bound of its own size: nothing
    # overflows before the scale is applied, and no bit of a small row is lost. Up to 2^-126 the bound also
    # takes the output's own step, 2^-149.
    qt, w, mag = _weight(n, k, bits, group, symmetric, seed=13)
    g = torch.Generator().manual_seed(14)
    x = torch.randn(m, k, generator=g).clamp_(-3, 3)
    size = torch.linspace(-140, 126, m).round()
    x = (x.double() * torch.exp2(size.double())[:, None]).float().to(DEV)
    bound = (x.double().abs() @ mag.t()) * ((3 * group + k / group + 4) * 2.0**-23 * (1 + 2.0**-7)) + 2.0**-148
    y, ref = ops.quant_linear(x, qt, None, torch.float32).double(), x.double() @ w.t()
    fits = ref.abs() < 3.4e38  # else the dense product is infinite as well
    assert bool(((y - ref).abs()[fits] <= bound[fits]).all()) and bool(torch.isinf(y[ref.abs() > 3.5e38]).all())


def test_swiglu_of_large_and_small_rows():
    # Each epilogue undoes the row's power of two: the one in the GEMM and the one in the reduction.
    for m, inter, k in ((33, 100, 1024), (300, 14336, 256)):
        qt, w, _ = _weight(2 * inter, k, 4, 64, True, seed=15)
        x = torch.randn(m, k, generator=torch.Generator().manual_seed(16)).to(DEV)
        y = ops.quant_linear_swiglu(x, qt, None, torch.float32)
        x[3] *= 2.0**-100  # exact
        x[5] *= 2.0**-70
        z = ops.quant_linear_swiglu(x, qt, None, torch.float32)
        keep = [i for i in range(m) if i not in (3, 5)]
        assert torch.equal(y[keep], z[keep])
        for r in (3, 5):  # silu(g) u is g u / 2 there
            t = (x[r].double() @ w.t()).view(inter // 4, 2, 4)
            ref = (t[:, 0] * t[:, 1] / 2).reshape(inter)
            assert float((z[r].double() - ref).abs().max()) <= 1e-5 * float(ref.abs().max()) + 2.0**-148


def test_partial_workspace_keeps_the_decode_passes():
    # Enough for the decode kernels' pieces and not for the GEMM's tiles: the chunks run as before.
    from llmopt.kernels import _lib

    lib = _lib.load_library()
    n, k, m = 512, 2048, 40
    qt, w, mag = _weight(n, k, 4, 64, True, seed=11)
    x = torch.randn(m, k, generator=torch.Generator().manual_seed(12)).to(DEV)
    full = ops.quant_linear(x, qt, None, torch.float32)
    for ws_bytes in (0, 4096, 3 * m * k * 2):
        y = torch.empty(m, n, device=DEV)
        ws = torch.empty(max(ws_bytes, 256), dtype=torch.uint8, device=DEV)
        rc = lib.llmopt_q_linear(x.data_ptr(), m, k, k, qt.qweight.data_ptr(), k // 2, qt.scales.data_ptr(),
                                 qt.zeros.data_ptr(), None, y.data_ptr(), n, n, _lib.DTYPE_CODES[torch.float32], 4,
                                 64, 1, 0, ws.data_ptr() if ws_bytes else None, ws_bytes,
                                 torch.cuda.current_stream().cuda_stream)
        assert rc == 0, lib.llmopt_q_last_error()
        assert float((y - full).abs().max()) <= 1e-5 * float(full.abs().max())


@pytest.mark.parametrize("m,inter,k", [(17, 128, 128), (33, 100, 1024), (65, 516, 2048), (500, 1024, 512), (300, 14336, 256)])
@pytest.mark.parametrize("with_bias", [False, True])
def test_swiglu_epilogue_and_reduction(m, inter, k, with_bias):
    # The activation in the GEMM's epilogue (no K split) and in its reduction (split): the product's fp32
    # error, through silu(g) u, whose slopes are at most 1.1 |u| and |g|, plus a few ulp of the hardware
    # exponential: within 2e-5 of the largest value.
    qt, w, _ = _weight(2 * inter, k, 4, 64, True, seed=m)
    g = torch.Generator().manual_seed(m)
    x = torch.randn(m, k, generator=g).to(DEV)
    bias = torch.randn(2 * inter, generator=g).to(DEV) if with_bias else None
    y = ops.quant_linear_swiglu(x, qt, bias, torch.float32)
    t = x.double() @ w.t()
    if bias is not None:
        t = t + bias.double()
    blocks = t.view(m, inter // 4, 2, 4)
    gate, up = blocks[:, :, 0].reshape(m, inter), blocks[:, :, 1].reshape(m, inter)
    ref = gate * torch.sigmoid(gate) * up
    assert y.shape == (m, inter)
    assert float((y.double() - ref).abs().max()) <= 2e-5 * float(ref.abs().max())
