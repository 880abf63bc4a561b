"""Latent decode in bf16 with one, two and four workgroups sharing a row block's value columns (by rows x heads), value widths that leave some of them without columns or with a part of
sixteen, and a context of more key splits than the sharing takes: against the oracle, 0.03 of the logits' spread (test_gpu_linasun.py's bar for bfloat16)."""
import pytest
import torch

import linasun_cases as LC
from oracle import linasun as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('rows', [1, 4, 9, 33])
@pytest.mark.parametrize('heads,dim,vdim,kv_rank', [(3, 64, 24, 64), (16, 128, 128, 512), (33, 64, 72, 128), (5, 192, 160, 256)])
def test_columns_shared_out(rows, heads, dim, vdim, kv_rank):
    from callireader_amd.modeling_decoder import LinasunForCausalLM
    cfg = LC.config(192, 150, [(LC.mixer(heads, dim, vdim, 64, kv_rank, dim ** -0.5), LC.moe(3, 2, 64, 1.5))])
    w = LC.weights(cfg, 51)
    m = LinasunForCausalLM.from_state_dict(w, cfg, dtype=torch.bfloat16, max_tokens=1400 if rows == 1 else 80, max_seqs=rows)
    toks = [LC.tokens(cfg, 1390 if rows == 1 else 3 + 11 * i % 70, seed=i) for i in range(rows)]
    m.step([(i, t[:-1], []) for i, t in enumerate(toks)])
    z = m.step([(i, t[-1:], [0]) for i, t in enumerate(toks)]).cpu()
    m.close()
    for i in sorted({0, rows // 2, rows - 1}):
        assert LC.rel(z[i:i + 1], O.forward(w, cfg, toks[i])[-1:]) < 0.03, i


@pytest.mark.parametrize('rows,keys', [(1, 5), (1, 700), (9, 40), (24, 600), (24, 700), (64, 20)])
@pytest.mark.parametrize('width,heads,dim,vdim,kv_rank', [(1024, 8, 128, 128, 256), (1152, 17, 64, 72, 128), (256, 3, 192, 128, 512), (2560, 16, 128, 128, 256)])
def test_weights_in_the_decode_layout_have_the_bits_of_rows(rows, keys, width, heads, dim, vdim, kv_rank, monkeypatch):
    """The projections into the latent and back with their weights fragment-ordered and as rows, and with that the attention with and without workgroups that fetch the output projection beside it (up
    to 128 workgroups of its own, and 144 with 24 rows of 700 keys, beside which the 10 MiB of the widest are left where they are): the same bits."""
    from callireader_amd.modeling_decoder import LinasunForCausalLM
    cfg = LC.config(width, 150, [(LC.mixer(heads, dim, vdim, 64, kv_rank, dim ** -0.5), LC.moe(3, 2, 64, 1.5))] * 2)
    w = LC.weights(cfg, 52)
    toks = [LC.tokens(cfg, keys + i % 3, seed=i) for i in range(rows)]
    got = []
    for layout in ('1', '0'):
        monkeypatch.setenv('CR_DECODE_LAYOUT', layout)
        m = LinasunForCausalLM.from_state_dict(w, cfg, dtype=torch.bfloat16, max_tokens=keys + 8, max_seqs=rows)
        m.step([(i, t[:-2], []) for i, t in enumerate(toks)])
        got.append(torch.stack([m.step([(i, [t[len(t) - 2 + k]], [0]) for i, t in enumerate(toks)]) for k in range(2)]).cpu())
        m.close()
    assert torch.isfinite(got[0]).all() and torch.equal(*got)
