"""Head dim 256 (bf16 / fp16) on the matrix-core scoring and attention kernels, against the oracle.

Tolerances are those of the other head dims on these kernels: scores rtol 1e-3 (float32 MFMA dot
products of exact 16-bit products, against the oracle's float32 folds), lse atol 1e-4, out atol
2e-4 (test_attention_gpu.py gives the derivation; it does not depend on the head dim)."""
import math

import pytest
import torch

from actkv.kernels.lse_attn import action_scores
from actkv.paged import PagedKVCache
from oracle import reference as ref

pytestmark = pytest.mark.gpu

D = 256


def _cache(lens, hkv, bs, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    nb = sum(math.ceil(n / bs) for n in lens) + 5
    cache = PagedKVCache(nb, bs, hkv, D, n_layers=1, dtype=dtype, device="cuda")
    cache.free = torch.randperm(nb, generator=g).tolist()
    for r, n in enumerate(lens):
        cache.append(r, torch.randn(1, n, hkv, D, generator=g).to(dtype).cuda(),
                     torch.randn(1, n, hkv, D, generator=g).to(dtype).cuda())
    return cache


@pytest.mark.parametrize("lens,hq,hkv,n_q,dtype,causal,bs,split", [
    ([700, 1500], 16, 8, 1, torch.bfloat16, False, 16, True),    # decode: 2 rows, one-wave ring
    ([1, 33, 640], 8, 8, 1, torch.float16, False, 32, True),     # G 1, a one-token request
    ([3000, 47], 32, 2, 2, torch.bfloat16, True, 16, True),      # G 16, 32 rows: one full tile
    ([3000, 47], 32, 2, 2, torch.float16, True, 16, False),      # the same in one pass
    ([900, 31], 16, 8, 24, torch.bfloat16, True, 16, True),      # 48 rows: 2-wave ring
    ([2000, 1337], 12, 4, 30, torch.bfloat16, True, 16, True),   # G 3, 90 rows: 4-wave ring
    ([640], 16, 8, 100, torch.float16, True, 64, True),          # 200 rows: two row groups
    ([640, 2200], 16, 8, 100, torch.bfloat16, False, 16, False),  # the same in one pass
    ([5000, 700], 8, 2, 40, torch.bfloat16, True, 256, True),    # chunk starts inside blocks
])
def test_attention_head_dim_256(monkeypatch, lens, hq, hkv, n_q, dtype, causal, bs, split):
    from actkv import _hip
    cache = _cache(lens, hkv, bs, dtype, seed=len(lens) * 100 + n_q + bs)
    reqs = list(range(len(lens)))
    g = torch.Generator().manual_seed(n_q + D)
    q = torch.randn(len(lens), n_q, hq, D, generator=g).to(dtype)
    kv_len = None
    if causal:
        kv_len = torch.stack([torch.randint(0, s + 8, (n_q,), generator=g) for s in lens]).to(torch.int32)
        kv_len[0, 0] = 0                                           # a query that sees nothing
    lib = _hip.lib()
    mb = max(len(t) for t in cache.tables.values())
    if split:
        assert lib.actkv_paged_attention_workspace_size(1, len(lens), n_q, hq, hkv, D, mb, bs) > 0
    else:
        monkeypatch.setattr(lib, "actkv_paged_attention_workspace_size", lambda *a: 0)
    out, lse = cache.decode_attention(reqs, q.cuda(), kv_len=None if kv_len is None else kv_len.cuda())
    want_out, want_lse = ref.paged_attention(q.float(), cache.kv[0].cpu().float(), [cache.tables[r] for r in reqs],
                                             lens, kv_len=None if kv_len is None else kv_len.tolist(), n_valid=None)
    torch.testing.assert_close(lse.cpu(), want_lse, rtol=0, atol=1e-4)
    torch.testing.assert_close(out.cpu(), want_out, rtol=0, atol=2e-4)
    if causal:
        assert float(lse[0, 0, 0]) == -math.inf and torch.equal(out[0, 0].cpu(), torch.zeros(hq, D))


@pytest.mark.parametrize("lens,hq,hkv,n_q,dtype,bs", [
    ([300, 77], 16, 8, 1, torch.bfloat16, 16),       # one action query, G 2
    ([1000, 17, 200], 16, 8, 64, torch.bfloat16, 16),   # 128 rows: two token groups of waves
    ([1000, 17], 16, 8, 65, torch.float16, 16),      # 130 rows: one token group
    ([520], 16, 8, 130, torch.bfloat16, 32),         # 260 rows: two launches
    ([300, 64], 8, 8, 70, torch.float16, 64),        # G 1
    ([300, 65], 12, 4, 40, torch.bfloat16, 16),      # G 3, laid out as 4 rows a query
    ([300, 63], 16, 2, 20, torch.bfloat16, 16),      # G 8
    ([300, 31], 24, 2, 20, torch.float16, 16),       # G 12, laid out as 16 rows a query
])
def test_scoring_head_dim_256(lens, hq, hkv, n_q, dtype, bs):
    cache = _cache(lens, hkv, bs, dtype, seed=hq + n_q)
    reqs = list(range(len(lens)))
    bt, seq = cache.block_table(reqs), cache.seq_tensor(reqs)
    kv0, tables = cache.kv[0].cpu(), [cache.tables[r] for r in reqs]
    g = torch.Generator().manual_seed(n_q)
    q = torch.randn(len(lens), n_q, hq, D, generator=g).to(dtype)
    lse = torch.stack([ref.decode_lse(q[:, n].float(), kv0, tables, lens) for n in range(n_q)], 1)
    n_valid = torch.tensor([max(1, n_q - 2 * i) for i in reqs], dtype=torch.int32)
    out0 = torch.rand(len(lens), hkv, bt.shape[1] * bs, generator=g)
    n0 = torch.tensor([2 * (i == 0) for i in reqs], dtype=torch.int32)
    for kv_len in (None, torch.stack([torch.randint(0, s + 3, (n_q,), generator=g) for s in lens]).to(torch.int32)):
        out_k, n_k, out_o, n_o = out0.cuda(), n0.cuda(), out0.clone(), n0.clone()
        action_scores(q.cuda(), cache.kv[0], bt, seq, lse.cuda(), out_k, n_k, n_valid=n_valid.cuda(),
                      kv_len=None if kv_len is None else kv_len.cuda())
        ref.action_scores_nfold(q.float(), kv0, tables, lens, lse, out_o, n_o, n_valid=n_valid, kv_len=kv_len)
        torch.testing.assert_close(out_k.cpu(), out_o, rtol=1e-3, atol=1e-6)
        assert torch.equal(n_k.cpu(), n_o)
