"""Decode attention at the edges of its work split, against the oracle's float64 attention.

With heads of 128 the grid of (sequence, KV head) pairs times context splits stays within one workgroup of
eight waves per CU (256 of them), and more than 256 pairs take four waves per workgroup up to a table of
1024 tokens; heads of 64 split as their smaller register count allows. Bounds as for every decode attention
output: the probabilities are rounded to the cache dtype (as the reference's are) and the output once to
the query dtype, 1e-2 for bf16 and 2e-3 for fp16."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from llmopt.cache import PagedKVCache
from llmopt.kernels import _lib, ops
from oracle import attention_oracle as ao

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
TOL = {torch.bfloat16: 1e-2, torch.float16: 2e-3}

# (sequences, heads, kv_heads, head_dim, longest context): pairs of 128, 129, 160 and 255 - 257, 264,
# 511 and 512; several splits capped (72 and 96 pairs over long contexts); 16 query heads per KV head;
# 257 and 264 pairs on both sides of a table of 64 tiles.
CASES = [
    (16, 16, 8, 128, 300), (129, 1, 1, 128, 300), (20, 32, 8, 128, 290), (255, 2, 1, 128, 150), (32, 8, 8, 128, 300),
    (257, 4, 1, 128, 150), (33, 32, 8, 128, 290), (73, 14, 7, 128, 150), (64, 8, 8, 128, 150), (9, 32, 8, 128, 1100),
    (12, 8, 8, 128, 1030), (20, 128, 8, 128, 290), (33, 128, 8, 128, 290), (20, 16, 8, 64, 290), (33, 16, 8, 64, 290),
    (257, 4, 1, 128, 1024), (257, 4, 1, 128, 1025), (33, 32, 8, 128, 1040),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_split_edges_match_oracle(case, dtype):
    seqs, heads, kv_heads, d, longest = CASES[case]
    rng = np.random.default_rng(case)
    ctx = rng.integers(1, longest + 1, size=seqs).astype(np.int32)
    ctx[0], ctx[seqs // 2] = longest, 0
    bs = 16
    width = -(-longest // bs)
    need = [-(-int(c) // bs) for c in ctx]
    perm = rng.permutation(sum(need) + 2).astype(np.int32)
    table = np.full((seqs, width), -1, dtype=np.int32)
    at = 0
    for s, n in enumerate(need):
        table[s, :n] = perm[at:at + n]
        at += n
    g = torch.Generator().manual_seed(case)
    cache = PagedKVCache(1, len(perm), bs, kv_heads, d, dtype=dtype, device=DEV)
    cache.key_cache.copy_(torch.randn(cache.key_cache.shape, generator=g).to(dtype))
    cache.value_cache.copy_(torch.randn(cache.value_cache.shape, generator=g).to(dtype))
    q = torch.randn(seqs, heads, d, generator=g).to(dtype)
    out = ops.paged_decode_attention(q.to(DEV), cache.key_cache[0], cache.value_cache[0],
                                     torch.from_numpy(table).to(DEV), torch.from_numpy(ctx).to(DEV), d ** -0.5)
    ref = ao.paged_decode_attention(q.float().numpy(), cache.key_cache.float().cpu().numpy(),
                                    cache.value_cache.float().cpu().numpy(), 0, table, ctx,
                                    cache_dtype="bfloat16" if dtype == torch.bfloat16 else "float16")
    got = out.float().cpu().numpy()
    assert np.all(got[ctx == 0] == 0)
    scale = float(np.abs(ref).max())
    assert float(np.abs(got - ref).max()) <= TOL[dtype] * scale


@pytest.mark.parametrize("pairs,splits", [(64, 4), (72, 3), (96, 2), (128, 2), (129, 1), (255, 1), (257, 1), (512, 1)])
def test_workspace_names_one_round(pairs, splits):
    """Contexts long enough for any split: 256 workgroups of eight waves at most, whatever the pairs."""
    need = _lib.load_library().llmopt_paged_attention_workspace(pairs, 4, 1, 128, 512, 16)
    assert need == (splits * pairs * 4 * 129 * 4 if splits > 1 else 0)
