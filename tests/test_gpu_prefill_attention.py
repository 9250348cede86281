"""The prefill attention kernel at the edges of its tiles: 128 query rows (tokens x heads of a KV head)
per workgroup, 32 per wave, 64 keys per tile. Against the same attention in float64 over the same cached
values; the bound is the coarser dtype's rounding of the probabilities and of the output (1e-2 of the
largest value in bf16, 2e-3 in fp16)."""

from __future__ import annotations

import pytest
import torch

from llmopt.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
TOL = {torch.bfloat16: 1e-2, torch.float16: 2e-3}


def _case(ctx, q_len, heads, kv_heads, d, bs, dtype, seed, spare=2):
    g = torch.Generator().manual_seed(seed)
    per = -(-max(ctx) // bs) + 1
    nb = len(ctx) * per + spare
    kc = torch.randn(nb, bs, kv_heads, d, generator=g).to(dtype).to(DEV)
    vc = torch.randn(nb, bs, kv_heads, d, generator=g).to(dtype).to(DEV)
    table = torch.randperm(nb, generator=g)[: len(ctx) * per].view(len(ctx), per).to(torch.int32)
    q = torch.randn(len(ctx), q_len, heads, d, generator=g).to(dtype).to(DEV).permute(0, 2, 1, 3)
    return q, kc, vc, table.to(DEV), torch.tensor(ctx, dtype=torch.int32, device=DEV)


def _reference(q, kc, vc, table, lens, bs, scale):
    seqs, heads, q_len, d = q.shape
    out = torch.zeros(seqs, heads, q_len, d, dtype=torch.float64, device=DEV)
    group = heads // kc.shape[2]
    for s in range(seqs):
        n = int(lens[s])
        t = torch.arange(n, device=DEV)
        ids = table[s].long()[t // bs]
        ok = ids >= 0
        rows = ids.clamp(min=0), t % bs
        k = kc[rows].double().permute(1, 0, 2).repeat_interleave(group, 0).contiguous()
        v = torch.where(ok[:, None, None], vc[rows].double(), 0.0).permute(1, 0, 2).repeat_interleave(group, 0)
        sc = torch.matmul(q[s].double().contiguous(), k.transpose(1, 2).contiguous()) * scale
        pos = n - q_len + torch.arange(q_len, device=DEV)
        sc = sc.masked_fill(~((t[None] <= pos[:, None]) & ok[None])[None], float("-inf"))
        out[s] = torch.matmul(torch.nan_to_num(torch.softmax(sc, -1)), v.contiguous())
    return out


def _rel(y, ref):
    return float((y.double() - ref).abs().max()) / max(float(ref.abs().max()), 1e-30)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("heads,kv_heads,d", [(8, 8, 128), (8, 4, 64), (8, 2, 128), (16, 2, 64), (16, 1, 128)])
@pytest.mark.parametrize("q_len", [2, 7, 8, 9, 31, 33, 65, 127, 129])
def test_query_edges(q_len, heads, kv_heads, d, dtype):
    ctx = [q_len, q_len + 63, q_len + 64, q_len + 1]  # no prefix, and prefixes around a key tile
    q, kc, vc, table, lens = _case(ctx, q_len, heads, kv_heads, d, 16, dtype, seed=q_len + heads)
    out = ops.paged_prefill_attention(q, kc, vc, table, lens, d**-0.5)
    assert _rel(out, _reference(q, kc, vc, table, lens, 16, d**-0.5)) <= TOL[dtype]


@pytest.mark.parametrize("bs", [1, 3, 8, 24, 64, 100])
def test_block_sizes_and_holes(bs):
    # Block sizes that are no powers of two, and holes: a -1 block and one past the pool.
    q, kc, vc, table, lens = _case([200, 90], 40, 8, 2, 128, bs, torch.bfloat16, seed=bs)
    table[0, 120 // bs] = -1
    table[1, 10 // bs] = -1
    out = ops.paged_prefill_attention(q, kc, vc, table, lens, 0.1)
    assert _rel(out, _reference(q, kc, vc, table, lens, bs, 0.1)) <= TOL[torch.bfloat16]
    past = table.clone()
    past[past < 0] = kc.shape[0] + 5
    assert torch.equal(out, ops.paged_prefill_attention(q, kc, vc, past, lens, 0.1))


def test_slots_that_are_no_keys_may_hold_anything():
    # Past each context the blocks hold NaN, and so does the hole's block 0: nothing of it reaches the
    # output. A context shorter than the chunk leaves its first tokens without keys: zeros.
    q, kc, vc, table, lens = _case([70, 20], 33, 8, 2, 128, 16, torch.bfloat16, seed=3)
    table[table == 0] = kc.shape[0] - 1
    for s, n in enumerate((70, 20)):
        for t in range(n, 80):
            kc[table[s, t // 16], t % 16] = float("nan")
            vc[table[s, t // 16], t % 16] = float("nan")
    kc[0], vc[0] = float("nan"), float("nan")
    table[0, 1] = -1
    out = ops.paged_prefill_attention(q, kc, vc, table, lens, 0.1)
    assert bool(torch.isfinite(out.float()).all())
    assert _rel(out, _reference(q, kc, vc, table, lens, 16, 0.1)) <= TOL[torch.bfloat16]
    assert int(torch.count_nonzero(out[1, :, :13])) == 0


@pytest.mark.parametrize("scale", [-0.2, 0.0])
def test_scales_that_are_not_positive(scale):
    q, kc, vc, table, lens = _case([150], 70, 8, 2, 64, 16, torch.float16, seed=4)
    out = ops.paged_prefill_attention(q, kc, vc, table, lens, scale)
    assert _rel(out, _reference(q, kc, vc, table, lens, 16, scale)) <= TOL[torch.float16]


@pytest.mark.parametrize("q_dtype", [torch.float32, torch.bfloat16])
def test_query_and_output_rows_off_alignment(q_dtype):
    # Query rows at an odd element offset are read element by element, with the aligned call's result.
    q, kc, vc, table, lens = _case([100, 64], 50, 8, 2, 128, 16, torch.bfloat16, seed=5)
    q = q.to(q_dtype)
    buf = torch.zeros(2, 50, 8 * 128 + 3, dtype=q_dtype, device=DEV)
    odd = buf[:, :, 1 : 1 + 8 * 128]
    odd.copy_(q.permute(0, 2, 1, 3).reshape(2, 50, 8 * 128))
    view = odd.as_strided((2, 8, 50, 128), (50 * buf.stride(1), 128, buf.stride(1), 1), odd.storage_offset())
    out = ops.paged_prefill_attention(q, kc, vc, table, lens, 0.1)
    assert torch.equal(out, ops.paged_prefill_attention(view, kc, vc, table, lens, 0.1))


def _stepwise(q, kc, vc, table, lens, bs, scale, step):
    """The same attention in float64 but for two roundings to the cache dtype: each probability's, relative
    to the running maximum of its row over steps of ``step`` keys, and the output's."""
    seqs, heads, q_len, d = q.shape
    out = torch.empty(seqs, heads, q_len, d, dtype=torch.float64, device=DEV)
    group = heads // kc.shape[2]
    for s in range(seqs):
        n = int(lens[s])
        t = torch.arange(n, device=DEV)
        rows = table[s].long()[t // bs], t % bs
        k, v = (c[rows].double().permute(1, 0, 2).repeat_interleave(group, 0).contiguous() for c in (kc, vc))
        sc = torch.matmul(q[s].double().contiguous(), k.transpose(1, 2).contiguous()) * scale
        pos = n - q_len + torch.arange(q_len, device=DEV)
        sc = sc.masked_fill((t[None] > pos[:, None])[None], float("-inf"))
        steps = torch.nn.functional.pad(sc, (0, -n % step), value=float("-inf")).unflatten(-1, (-1, step))
        top = steps.amax(-1).cummax(-1).values
        p = torch.exp(steps - top[..., None])
        back = torch.exp(top - top[..., -1:])[..., None]
        o = torch.matmul((p.to(q.dtype).double() * back).flatten(-2)[..., :n].contiguous(), v)
        out[s] = (o / (p * back).sum((-2, -1))[..., None]).to(q.dtype).double()
    return out


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_error_of_rounded_probabilities(dtype):
    # Prompts of 512 tokens: no further from float64 than the roundings alone put steps of 16 keys (half a
    # percent for what 8192 rows of random roundings differ by).
    q, kc, vc, table, lens = _case([512, 512], 512, 8, 2, 128, 16, dtype, seed=6)
    ref = _reference(q, kc, vc, table, lens, 16, 128**-0.5)
    out = ops.paged_prefill_attention(q, kc, vc, table, lens, 128**-0.5)
    steps = _stepwise(q, kc, vc, table, lens, 16, 128**-0.5, 16)
    assert float((out.double() - ref).norm()) <= 1.005 * float((steps - ref).norm())
