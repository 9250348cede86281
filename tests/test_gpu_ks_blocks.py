"""The K-sliced decode kernel with three token blocks (33 - 48 tokens, nibble and byte codes) and its
neighbours with two and four, against the float64 product of the exact weight. Bound: the operands are
exact (code plus offset in bf16 / fp16), so K fp32 additions of 2^-23 each over the magnitudes summed, the
offset's (up to 128 + q in bf16, 1024 + q in fp16) included, and one rounding of the output."""

from __future__ import annotations

import pytest
import torch

from llmopt.kernels import ops
from llmopt.quantization import QuantizedTensor

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype,offset,ulp", [(torch.bfloat16, 128, 2.0**-8), (torch.float16, 1024, 2.0**-11)])
@pytest.mark.parametrize("bits,group,symmetric", [(4, 128, False), (4, 256, True), (8, 128, True)])
@pytest.mark.parametrize("m", [32, 33, 47, 48, 49, 64])
def test_token_blocks(m, bits, group, symmetric, dtype, offset, ulp):
    n, k = 200, 4096
    g = torch.Generator().manual_seed(m + bits)
    codes = torch.randint(0, 1 << bits, (n, k), generator=g)
    scales = torch.rand(n, k // group, generator=g) * 0.01 + 0.002
    zeros = torch.randint(0, 1 << bits, scales.shape, generator=g).float() * (not symmetric)
    points = torch.full_like(scales, float(1 << (bits - 1))) if symmetric else zeros
    c8 = codes.to(torch.uint8)
    q = (codes - 128).to(torch.int8) if bits == 8 else c8[:, 0::2] | (c8[:, 1::2] << 4)
    qt = QuantizedTensor(q.contiguous().to(DEV), scales.to(DEV), zeros.to(DEV), bits, group, symmetric, (n, k))
    w = ((codes.view(n, -1, group).double() - points.double()[..., None]) * scales.double()[..., None]).view(n, k)
    mag = ((codes.view(n, -1, group).double() + offset + 128) * scales.double()[..., None]).view(n, k)
    x = torch.randn(m, k, generator=g).to(dtype).to(DEV)
    y = ops.quant_linear(x, qt, None, dtype)
    ref = x.double() @ w.t().to(DEV)
    bound = (x.double().abs() @ mag.t().to(DEV)) * (2 * group * 2.0**-23) + ref.abs() * ulp
    assert bool(((y.double() - ref).abs() <= bound).all())
