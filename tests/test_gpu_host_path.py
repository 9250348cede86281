"""The native host path of the linears against the general one: the same bits for every plain call, the
general path (conversions, broadcasts, torch's errors) for every other form, the current stream, no
alias between results, and replays of a captured call."""

from __future__ import annotations

import pytest
import torch
from torch import nn

from llmopt.kernels import ops
from llmopt.quantization import FusedQuantLinear, QuantLinear, QuantSwiGLU, RoundToNearestQuantizer

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _module(n, k, bits, group, symmetric, dtype, bias, seed=0):
    g = torch.Generator().manual_seed(seed)
    linear = nn.Linear(k, n, bias=bias, dtype=dtype)
    with torch.no_grad():
        linear.weight.copy_(torch.randn(n, k, generator=g) * 0.02)
    qt = RoundToNearestQuantizer(bits, group, symmetric).quantize(linear.weight.detach().float())
    return QuantLinear.from_float(linear, qt, compute_dtype=dtype).to(DEV)


def _general(m, x):
    return ops.quant_linear(x, m.quantized_tensor(), m.bias, m.config.compute_dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("bits,group,symmetric,bias", [(4, 128, False, True), (4, 64, True, False),
                                                       (8, 128, True, True), (8, 32, False, False), (2, 256, True, True)])
@pytest.mark.parametrize("shape", [(256,), (1, 256), (3, 256), (2, 5, 256), (70, 256), (1100, 256)])
def test_same_bits_as_the_general_path(shape, bits, group, symmetric, bias, dtype):
    m = _module(96, 256, bits, group, symmetric, dtype, bias)
    x = torch.randn(*shape, generator=torch.Generator().manual_seed(1)).to(dtype).to(DEV)
    y = ops.module_linear(x, m, 96)
    assert y is not None and y.shape == (*shape[:-1], 96) and y.dtype == dtype and not y.requires_grad
    assert torch.equal(y, _general(m, x)) and torch.equal(m(x), y)


@pytest.mark.parametrize("m_tokens", [1, 40, 300])
def test_fused_modules(m_tokens):
    parts = [_module(n, 512, 4, 128, False, torch.bfloat16, False, seed=n) for n in (64, 32, 32)]
    x = torch.randn(m_tokens, 512, device=DEV).to(torch.bfloat16)
    fused = FusedQuantLinear(parts)
    y = ops.quant_linear(x, fused.quantized_tensor(), fused.bias, torch.bfloat16)
    assert all(torch.equal(a, b) for a, b in zip(fused(x), torch.split(y, [64, 32, 32], dim=-1)))
    gate, up = (_module(64, 512, 4, 128, False, torch.bfloat16, True, seed=s) for s in (1, 2))
    swiglu = QuantSwiGLU(gate, up)
    want = ops.quant_linear_swiglu(x, swiglu.quantized_tensor(), swiglu.bias, torch.bfloat16)
    assert ops.module_linear(x, swiglu, 128, swiglu=True) is not None and torch.equal(swiglu(x), want)


def test_other_forms_take_the_general_path():
    m = _module(64, 256, 4, 128, False, torch.bfloat16, True)
    x = torch.randn(6, 256, device=DEV).to(torch.bfloat16)
    assert ops.module_linear(x[::2], m, 64) is None  # strided rows
    assert torch.equal(m(x[::2]), m(x)[::2])
    assert ops.module_linear(x.t().contiguous().t(), m, 64) is None
    assert ops.module_linear(x[:0], m, 64) is None and m(x[:0]).shape == (0, 64)
    sub = x.as_subclass(type("Sub", (torch.Tensor,), {}))
    assert ops.module_linear(sub, m, 64) is None and torch.equal(m(sub), m(x))
    for bad, exc in ((x.float(), RuntimeError), (x[:, :128], RuntimeError), (x.cpu(), RuntimeError)):
        if bad.is_cuda:
            assert ops.module_linear(bad, m, 64) is None
            with pytest.raises(exc):
                m(bad)
    y = m(x)
    m.scales = m.scales.to(torch.float16).float()[:, :1].expand(64, 2)  # a broadcast table
    assert ops.module_linear(x, m, 64) is None
    assert torch.equal(m(x), _general(m, x)) and y.shape == (6, 64)
    m.scales = m.scales.contiguous()[:32]
    assert ops.module_linear(x, m, 64) is None
    with pytest.raises(RuntimeError):
        m(x)
    m.config.compute_dtype = torch.float64
    assert ops.module_linear(x, m, 64) is None
    with pytest.raises((RuntimeError, TypeError)):
        m(x)


@pytest.mark.parametrize("fused", [False, True])
def test_out_of_memory_is_torchs_own_error(fused):
    # The output (512 MB) does not fit the share of the card that this process may take: callers catch
    # torch.OutOfMemoryError, drop the batch and go on.
    m = _module(4096, 256, 4, 128, False, torch.bfloat16, False)
    m = FusedQuantLinear([m]) if fused else m
    x = torch.zeros(65536, 256, dtype=torch.bfloat16, device=DEV)
    small = m(x[:8])
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (128 << 20)) / total)
    try:
        with pytest.raises(torch.OutOfMemoryError):
            m(x)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    again = m(x[:8])
    assert all(torch.equal(a, b) for a, b in zip(again, small))


def test_a_subclass_keeps_its_own_weight():
    class Halved(QuantLinear):
        def quantized_tensor(self):
            t = super().quantized_tensor()
            return type(t)(t.qweight, t.scales * 0.5, t.zeros, t.bits, t.group_size, t.symmetric, t.shape)

    m = _module(64, 256, 4, 128, False, torch.float32, False)
    x = torch.randn(3, 256, device=DEV)
    y = m(x)
    m.__class__ = Halved
    assert torch.equal(m(x), y * 0.5)


def test_calls_follow_the_work_before_them_on_a_side_stream():
    # Milliseconds of products make the first input, then each call's input is the last one's output: a
    # launch on another stream, or one that reads a buffer too early or a reused one, changes the end.
    m = _module(4096, 4096, 4, 128, False, torch.bfloat16, False)
    a = torch.randn(4096, 4096, generator=torch.Generator().manual_seed(3)).to(torch.bfloat16).to(DEV) / 64

    def chain():
        t = a
        for _ in range(20):
            t = t @ a
        y, outs = t[:1] * 1.0, []
        for i in range(20):
            y = m(y) * (0.75 + 0.01 * i)
            outs.append(y)
        return torch.cat(outs)

    want = chain()
    assert bool(torch.isfinite(want.float()).all()) and len(set(want.float().norm(dim=1).tolist())) == 20
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert torch.cuda.current_stream().cuda_stream == side.cuda_stream
        got = chain()
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(got, want)


def test_capture_and_separate_outputs():
    m = _module(512, 4096, 4, 128, False, torch.bfloat16, False)
    x = torch.randn(1, 4096, device=DEV).to(torch.bfloat16)
    want = m(x)
    a, b = m(x), m(x * 2)
    assert a.data_ptr() != b.data_ptr() and torch.equal(a, want)
    static = x.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = m(static)
    for scale in (1.0, -3.0, 0.5):
        static.copy_(x * scale)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, m(x * scale))
