"""The class rows of a tile are merged by workgroups of four heads, beside the one that redoes flagged query blocks: head counts around multiples of four, key counts with the merge's
own number of partials (33) and others, a flagged block in the last head.  Reference: the same arithmetic in fp32 with the bf16 rounding points; bounds of test_gpu_ops.py."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('H', [1, 3, 4, 5, 16])
@pytest.mark.parametrize('S', [385, 1025])
def test_class_rows_and_flagged_blocks(H, S):
    from callireader_amd import engine as E
    g = torch.Generator().manual_seed(H * S)
    rb = lambda t: t.to(torch.bfloat16).float()
    Bn, D = 3, 64
    qkv = torch.randn(Bn, S, 3 * H * D, generator=g).to(torch.bfloat16)
    spike = torch.zeros(D, dtype=torch.bfloat16)
    spike[0] = 32.0
    last = (H - 1) * D
    qkv[1, 200, last:last + D] = spike                       # scores of 0 against the class key and 128 against key 7: past the lean sweep
    qkv[1, 0, H * D + last:H * D + last + D] = 0
    qkv[1, 7, H * D + last:H * D + last + D] = spike
    o = torch.full((Bn, S, H * D), float('nan'), device='cuda', dtype=torch.bfloat16)
    x = qkv.cuda()
    strides = [S * 3 * H * D, 3 * H * D, D] * 3 + [S * H * D, H * D, D]
    E.op_attention(x, x[..., H * D:], x[..., 2 * H * D:], o, strides, Bn, H, S, S, D, q_prescale=0.125)
    q, k, v = (t.float().view(Bn, S, H, D).transpose(1, 2) for t in qkv.split(H * D, -1))
    want = rb(rb(torch.softmax(rb(rb(q * 0.125) @ k.transpose(-1, -2)), -1)) @ v).transpose(1, 2).reshape(Bn, S, H * D)
    torch.testing.assert_close(o.float().cpu(), want, rtol=1.6e-2, atol=1.5e-2)
