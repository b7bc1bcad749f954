"""Scoring over requests of very different lengths and query counts in one launch: every token
range of every request is taken exactly once, whatever the number of requests, head packs per
launch and empty requests."""
import math
import random

import pytest
import torch

from actkv.kernels.lse_attn import action_scores
from actkv.paged import PagedKVCache
from oracle import reference as ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_req,layers,hq,hkv,d,n_q,seed", [
    (2, 3, 16, 8, 64, 40, 0),      # 80 rows, 4 heads a workgroup: packs that do not divide by 8
    (5, 2, 16, 8, 64, 5, 1),       # 10 rows, 8 heads a workgroup: one pack
    (7, 2, 8, 4, 128, 150, 2),     # 300 rows, K-slice kernel, 4 heads: not a multiple of 8
    (9, 1, 16, 8, 128, 260, 3),    # 520 rows with counts per request: K-slice, two launches
    (64, 1, 8, 8, 64, 20, 4),      # as many requests as lanes
    (65, 1, 8, 8, 64, 20, 5),      # one more: plain order
    (4, 1, 16, 8, 256, 30, 6),     # head dim 256, 60 rows
])
def test_every_range_is_scored_once(n_req, layers, hq, hkv, d, n_q, seed):
    rnd = random.Random(seed)
    g = torch.Generator().manual_seed(seed)
    bs, dt = 16, torch.bfloat16
    lens = [rnd.choice([0, 1, rnd.randint(2, 90), rnd.randint(90, 2600 if n_req < 20 else 300)]) for _ in range(n_req)]
    lens[rnd.randrange(n_req)] = 2601 if n_req < 20 else 301
    nb = sum(math.ceil(s / bs) for s in lens) + 2
    cache = PagedKVCache(nb, bs, hkv, d, n_layers=layers, dtype=dt, device="cuda")
    cache.free = torch.randperm(nb, generator=g).tolist()
    for r, s in enumerate(lens):
        x = torch.randn(layers, s, hkv, d, generator=g).to(dt).cuda()
        cache.append(r, x, x)
    reqs = list(range(n_req))
    bt, seq = cache.block_table(reqs), cache.seq_tensor(reqs)
    q = torch.randn(layers, n_req, n_q, hq, d, generator=g).to(dt)
    lse = torch.full((layers, n_req, n_q, hq), 7.0) + torch.rand(layers, n_req, n_q, hq, generator=g)
    n_valid = torch.tensor([rnd.choice([0, 1, n_q // 2, n_q]) for _ in reqs], dtype=torch.int32)
    n_valid[lens.index(max(lens))] = n_q
    width = bt.shape[1] * bs
    out0 = torch.rand(layers, n_req, hkv, width, generator=g)
    n0 = torch.tensor([i % 3 for i in reqs], dtype=torch.int32)
    out, n_seen = out0.cuda(), n0.cuda()
    action_scores(q.cuda(), cache.kv, bt, seq, lse.cuda(), out, n_seen, n_valid=n_valid.cuda())
    for l in range(layers):
        want, n_want = out0[l].clone(), n0.clone()
        ref.action_scores_nfold(q[l].float(), cache.kv[l].cpu().float(), [cache.tables[r] for r in reqs], lens,
                                lse[l], want, n_want, n_valid=n_valid)
        # float32 dot products of exact 16-bit products in another order: the scoring tests' bound
        torch.testing.assert_close(out[l].cpu(), want, rtol=1e-3, atol=1e-6)
        assert torch.equal(n_seen.cpu(), n_want)
