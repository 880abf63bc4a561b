"""Causal attention deals its workgroups out by XCD: where XCDs get whole heads, eight of them together with the longest query blocks first.  Every (batch, head, block) is computed once and
wherever it runs: a launch of many heads against each head launched alone, bit for bit, at counts of heads that leave a smaller last group, a single one, or no whole heads for an XCD."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('B,H,S', [(1, 8, 129), (3, 8, 300), (2, 48, 257), (8, 17, 130), (5, 7, 300)])
def test_every_block_once(B, H, S):
    from callireader_amd import engine as E
    D = 128
    g = torch.Generator(device='cuda').manual_seed(B * 100 + H)
    q, k, v = (torch.randn(B, S, H, D, device='cuda', generator=g).to(torch.bfloat16) for _ in range(3))
    o, one = torch.zeros_like(q), torch.zeros_like(q)
    st = [S * H * D, H * D, D] * 4
    E.op_attention(q, k, v, o, st, B, H, S, S, D, causal=True, s_div=math.sqrt(D))
    for b in range(B):
        for h in range(H):
            E.op_attention(q[b, :, h], k[b, :, h], v[b, :, h], one[b, :, h], st, 1, 1, S, S, D, causal=True, s_div=math.sqrt(D))
    torch.cuda.synchronize()
    assert torch.equal(o, one) and bool(o.float().abs().sum(-1).min() > 0)
