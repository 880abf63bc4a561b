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


@pytest.mark.parametrize('D,H,G,softcap,lens', [(128, 16, 4, 50.0, (300, 129, 1, 640)),             # 64 heads in all, 8 an XCD
                                                (128, 48, 48, 0.0, (257, 130, 384)),                # 144: 18 an XCD, the last group of two
                                                (64, 8, 2, 20.0, (128, 127, 129, 1, 255, 500, 64, 383, 256)),      # 72: nine
                                                (64, 17, 17, 0.0, (300, 200)),                      # 34: no whole heads for an XCD
                                                (256, 8, 8, 30.0, (200, 333, 129))])
def test_segments_of_unequal_length(D, H, G, softcap, lens):
    """The described decoders' instances: 32-bit scores, capped or not, several prompts in a launch of which some have fewer query blocks, a few of them behind cached keys."""
    from callireader_amd import engine as E
    g = torch.Generator(device='cuda').manual_seed(D + H)
    before = [37 * i % 90 for i in range(len(lens))]           # keys ahead of a segment's own
    segs, row, key = [], 0, 0
    for n, p in zip(lens, before):
        segs.append((row, n, p, key))
        row += n
        key += p + n
    q = torch.randn(row, H, D, device='cuda', generator=g).to(torch.bfloat16)
    k, v = (torch.randn(key, G, D, device='cuda', generator=g).to(torch.bfloat16) for _ in range(2))
    vdim = D - 3 if D == 64 else D
    o = E.op_prompt_attention(q, k, v, segs, D ** -0.5, softcap, 0.7, vdim)
    one = torch.zeros_like(o)
    for s in segs:
        for h in range(H):
            one[s[0]:s[0] + s[1], h] = E.op_prompt_attention(q[:, h:h + 1].contiguous(), k[:, h * G // H, None].contiguous(), v[:, h * G // H, None].contiguous(), [s], D ** -0.5, softcap, 0.7,
                                                             vdim)[s[0]:s[0] + s[1], 0]
    assert torch.equal(o, one) and bool(o.float().abs().sum(-1).min() > 0)
    for r, n, p, kr in segs[:2]:                              # and against float32
        K, V = (t[kr:kr + p + n].float().repeat_interleave(H // G, 1).transpose(0, 1).contiguous() for t in (k, v))
        z = q[r:r + n].float().transpose(0, 1) @ K.transpose(1, 2).contiguous() * D ** -0.5
        z = softcap * torch.tanh(z / softcap) if softcap else z
        z = z.masked_fill(torch.arange(p + n, device='cuda')[None] > torch.arange(n, device='cuda')[:, None] + p, -math.inf)
        ref = 0.7 * (torch.softmax(z, -1) @ V)[..., :vdim].transpose(0, 1)
        assert float((o[r:r + n].float() - ref).norm() / ref.norm()) < 4e-3      # (bf16 results: 2^-9 at most, a third of it on average)
