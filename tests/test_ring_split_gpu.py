"""Ring attention: many token chunks per pair (merged 16 rows at a time) and rows whose maximum
keeps rising (the reference the probabilities are taken against moves, or lags by less than 8)."""
import math

import pytest
import torch

from actkv import _hip
from actkv.paged import PagedKVCache
from oracle import reference as ref

pytestmark = pytest.mark.gpu


def _cache(lens, hkv, d, dtype, rise):
    g = torch.Generator().manual_seed(d + len(lens))
    bs = 16
    nb = sum(-(-s // bs) for s in lens) + 3
    cache = PagedKVCache(nb, bs, hkv, d, dtype=dtype, device="cuda")
    cache.free = torch.randperm(nb, generator=g).tolist()
    u = torch.ones(d) / math.sqrt(d)
    for r, s in enumerate(lens):
        k = torch.randn(1, s, hkv, d, generator=g)
        k += (rise * torch.arange(s) / s).view(1, s, 1, 1) * u      # logits climb by about `rise`
        v = torch.randn(1, s, hkv, d, generator=g)
        cache.append(r, k.to(dtype).cuda(), v.to(dtype).cuda())
    return cache, u


@pytest.mark.parametrize("rise", [0.0, 60.0])
@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("lens,n_q,dtype,causal", [
    ([12011], 20, torch.bfloat16, False),            # one pair, 80 rows: more than 16 chunks
    ([9001, 333], 90, torch.float16, True),          # 360 rows: two row groups at 8 waves
    ([700, 257], 9, torch.bfloat16, True),           # 36 rows, chunks end inside a stage
])
def test_ring_chunks_and_rising_maxima(monkeypatch, lens, n_q, dtype, causal, d, rise):
    cache, u = _cache(lens, 1, d, dtype, rise)
    reqs = list(range(len(lens)))
    g = torch.Generator().manual_seed(n_q)
    q = (torch.randn(len(lens), n_q, 4, d, generator=g) + u * math.sqrt(d)).to(dtype)
    kv_len = None
    if causal:
        kv_len = torch.tensor([[max(0, s - n_q + j + 1) for j in range(n_q)] for s in lens], dtype=torch.int32)
    call = lambda: cache.decode_attention(reqs, q.cuda(), kv_len=None if kv_len is None else kv_len.cuda())
    lib = _hip.lib()
    if len(lens) == 1:
        mb = len(cache.tables[0])
        assert lib.actkv_paged_attention_workspace_size(1, 1, n_q, 4, 1, d, mb, 16) >= 17 * n_q * 4 * (d + 2) * 4
    out, lse = call()
    monkeypatch.setattr(lib, "actkv_paged_attention_workspace_size", lambda *a: 0)
    out1, lse1 = call()
    want_out, want_lse = ref.paged_attention(q.float(), cache.kv[0].cpu().float(), [cache.tables[r] for r in reqs],
                                             lens, kv_len=None if kv_len is None else kv_len.tolist(), n_valid=None)
    # probabilities carry 16 bits or more (2^-17 each way) against values of order 1
    for o, l in ((out, lse), (out1, lse1)):
        torch.testing.assert_close(l.cpu(), want_lse, rtol=0, atol=1e-4)
        torch.testing.assert_close(o.cpu(), want_out, rtol=0, atol=2e-4)
