"""The register-dequant GEMM's tile heights between 128 and 256 tokens (160, 192, 224), which the plan picks
for ragged batches over wide weights: every output against the float64 product of the rounded dequantized
weight. Bound: K fp32 additions of exact products (each at most 2^-23 of the magnitudes summed) and one
rounding of the output (ROUND: twice 2^-9 in bf16, 2^-12 in fp16). With SwiGLU: those errors of gate and up
through silu(g) u, whose slopes are at most 1.1 |u| and |silu(g)|, and the roundings of silu(g) and of the
product."""

from __future__ import annotations

import pytest
import torch

from llmopt.kernels import ops
from llmopt.kernels._lib import ALGO_PREFILL
from llmopt.quantization import QuantizedTensor, dequantize

pytestmark = pytest.mark.gpu
DEV = "cuda"
ROUND = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11}


def _weight(n, k, group, symmetric, seed):
    g = torch.Generator().manual_seed(seed)
    q = torch.randint(0, 256, (n, k // 2), generator=g, dtype=torch.uint8)
    s = torch.rand(n, k // group, generator=g) * 0.01 + 0.002
    z = torch.randint(0, 16, s.shape, generator=g).float() * (not symmetric)
    return QuantizedTensor(q.to(DEV), s.to(DEV), z.to(DEV), 4, group, symmetric, (n, k))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("group,symmetric", [(128, False), (64, True)])
@pytest.mark.parametrize("m", [257, 319, 320, 321, 384, 385, 448, 449, 600, 1100])
def test_heights(m, group, symmetric, dtype):
    n, k = 28672 - 40, 256
    qt = _weight(n, k, group, symmetric, seed=m)
    x = torch.randn(m, k, generator=torch.Generator().manual_seed(1)).to(dtype).to(DEV)
    w = dequantize(qt, dtype).double()
    y = ops.quant_linear(x, qt, None, dtype, algo=ALGO_PREFILL)
    ref = x.double() @ w.t()
    bound = (x.double().abs() @ w.abs().t()) * (k * 2.0**-23) + ref.abs() * ROUND[dtype]
    assert bool(((y.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("m", [290, 380, 440])
def test_heights_with_swiglu(m):
    inter, k = 14336, 256
    qt = _weight(2 * inter, k, 128, False, seed=m)
    x = torch.randn(m, k, generator=torch.Generator().manual_seed(2)).to(torch.bfloat16).to(DEV)
    y = ops.quant_linear_swiglu(x, qt, None, torch.bfloat16)
    w = dequantize(qt, torch.bfloat16).double()
    t = x.double() @ w.t()
    off = (x.double().abs() @ w.abs().t()) * (k * 2.0**-23) + t.abs() * ROUND[torch.bfloat16]
    gate, up, d_gate, d_up = [v.view(m, inter // 4, 2, 4)[:, :, i].reshape(m, inter) for v in (t, off) for i in (0, 1)]
    silu = gate * torch.sigmoid(gate)
    ref = silu * up
    bound = 1.1 * d_gate * up.abs() + silu.abs() * d_up + 1.1 * d_gate * d_up + 2 * ROUND[torch.bfloat16] * ref.abs()
    assert bool(((y.double() - ref).abs() <= bound).all())
