"""LRFU action scores of 8 heads, four tokens per thread: every remainder of the length and of the
protected prefix, both reductions, and rows that are not 16-byte aligned (one token per thread)."""
import pytest
import torch

from actkv.kernels.lrfu import lrfu_update

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("reduce", ["mean", "max"])
@pytest.mark.parametrize("width,off", [(1100, 0), (1101, 0), (1104, 1), (1104, 2)])
def test_aligned_and_unaligned_rows_agree(width, off, reduce):
    seqs, prots = [1, 3, 5, 30, 1027, 1090], [0, 2, 5, 7, 1, 1089]
    R, L, H = len(seqs), 2, 8
    g = torch.Generator().manual_seed(width + off)
    buf = torch.rand(L * R * H * width + 8, generator=g).cuda()
    scores = buf[off:off + L * R * H * width].view(L, R, H, width)
    # a copy whose rows start 4 bytes off takes the one-token kernel whatever `scores` takes
    odd = torch.empty(L, R, H, 1201, device="cuda")[..., 1:1 + width]
    odd.copy_(scores)
    ks = torch.rand(L, R, 1100, generator=g).cuda()
    ks1, ks2 = ks.clone(), ks.clone()
    hit1 = lrfu_update(scores, ks1, seqs, prots, decay=0.5, top_p=0.8, head_reduce=reduce, return_hits=True)
    hit2 = lrfu_update(odd, ks2, seqs, prots, decay=0.5, top_p=0.8, head_reduce=reduce, return_hits=True)
    assert torch.equal(ks1, ks2)
    for r, (s, p) in enumerate(zip(seqs, prots)):
        assert torch.equal(hit1[:, r, p:s], hit2[:, r, p:s])
        if p < s:
            want = scores[:, r, :, p:s].cpu()
            act = want.mean(1) if reduce == "mean" else want.amax(1)
            got = ks1[:, r, p:s].cpu() - 0.5 * ks[:, r, p:s].cpu()
            h = hit1[:, r, p:s].cpu()
            # one rounding of the sum and one of the halved score: 2^-23 of values below 2
            torch.testing.assert_close(got[h], act[h], rtol=0, atol=1e-6)
            assert torch.equal(got[~h], torch.zeros_like(got[~h]))
