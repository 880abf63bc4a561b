"""One launch for a decode step's attention and retention (lm_mix.hip): key counts around its 32-key blocks, 64-key tiles and 256-key splits, groups of query heads from one to the most a
workgroup takes, heads of 64 and 128, rotations whose halves are no multiple of eight, value sizes that no vector divides."""
import pytest
import torch

import lugasun_cases as LC
from oracle import lugasun as O

pytestmark = pytest.mark.gpu
F32, BF16 = torch.float32, torch.bfloat16
WIDTH = 512      # (a bf16 layer of fewer than 256 columns has no K-slices and keeps the separate kernels)
LENS = [1, 2, 31, 32, 33, 63, 64, 65, 96, 254, 255, 256, 257, 511, 513]
LAYERS = {
    'group4_128': LC.layer(LC.heads(8, 2, 128, 128, 4096, softcap=20.0), LC.ret(64, 64, (0.97, 0.9)), 64),
    'group1_64': LC.layer(LC.heads(3, 3, 50, 50, 4096, rot=(100.0, 36)), LC.ret(100, 300, (0.95,), rot=(100.0, 12)), None),
    'group32_128': LC.layer(LC.heads(32, 1, 72, 70, 4096), LC.ret(40, 33, (0.9, 0.99, 0.5)), None),
    'chunks': LC.layer(LC.heads(4, 1, 64, 64, 256), LC.ret(128, 64, (0.99,)), 64),
}


@pytest.mark.parametrize('dtype', [F32, BF16])
@pytest.mark.parametrize('name', LAYERS)
def test_rows_of_every_length_together_and_alone(name, dtype):
    """Against the oracle, and a row's bits are the same whatever longer or shorter rows it is decoded with."""
    from callireader_amd.modeling_decoder import LugasunForCausalLM
    cfg = LC.config(WIDTH, 60, [LAYERS[name]], side=8)
    w = LC.weights(cfg, 31, qk_gain=1.5 if dtype == F32 else 1.0)
    m = LugasunForCausalLM.from_state_dict(w, cfg, dtype=dtype, max_tokens=640, max_seqs=len(LENS))
    toks = [LC.tokens(cfg, n + 3, seed=n) for n in LENS]

    def run(which):
        for i in which:                                       # (a prompt alone, so that its bits are given)
            m.step([(i, toks[i][:LENS[i]], [])])
        z = torch.stack([m.step([(i, [toks[i][LENS[i] + k]], [0]) for i in which]) for k in range(3)], 1).cpu()
        for i in which:
            m.end(i)
        return z
    together = run(range(len(LENS)))
    for i, n in enumerate(LENS):
        assert LC.close(together[i], O.forward(w, cfg, toks[i])[n:], dtype), n
    for i in (0, 3, 6, 9, 12):
        assert torch.equal(run([i])[0], together[i]), LENS[i]
    m.close()


@pytest.mark.parametrize('dtype', [F32, BF16])
@pytest.mark.parametrize('name', LAYERS)
def test_one_launch_has_the_bits_of_the_separate_ones(name, dtype, monkeypatch):
    """Against the kernels it stands for (row kernel, split attention, retention with its merge), which other sizes take: logits, and what later steps read from caches and states.  Sharp scores move
    the reference point of the softmax from tile to tile, in some of a unit's queries and not in others."""
    from callireader_amd.modeling_decoder import LugasunForCausalLM
    cfg = LC.config(WIDTH, 60, [LAYERS[name], LAYERS[name]], side=8)
    w = LC.weights(cfg, 33, qk_gain=1.5)
    toks = [LC.tokens(cfg, n + 4, seed=n) for n in LENS]
    got = []
    for joined in ('1', '0'):
        monkeypatch.setenv('CR_DECODE_JOINED', joined)
        m = LugasunForCausalLM.from_state_dict(w, cfg, dtype=dtype, max_tokens=640, max_seqs=len(LENS))
        for i, n in enumerate(LENS):
            m.step([(i, toks[i][:n], [])])
        # (five rows at a time: more would be too many workgroups for one launch in float32)
        got.append(torch.stack([torch.cat([m.step([(i, [toks[i][LENS[i] + k]], [0]) for i in range(j, j + 5)]) for j in range(0, len(LENS), 5)]) for k in range(4)]).cpu())
        m.close()
    assert torch.equal(*got), [(int(k), LENS[int(i)]) for k, i in (got[0] != got[1]).any(-1).nonzero()]


@pytest.mark.parametrize('dtype', [F32, BF16])
@pytest.mark.parametrize('width', [200, 1024, 2048])
def test_residual_updates_inside_the_next_product(width, dtype):
    """One to a few rows leave each residual update to the product behind it (lm_ahead.hip), more rows take a launch for it: the same bits, with and without norms on the way, at the entry of
    a looped span and ahead of the token side."""
    from callireader_amd.modeling_decoder import LugasunForCausalLM
    cfg = LC.config(width, 90, [LC.layer(LC.heads(2, 1, 64, 64, 64), LC.ret(64, 64, (0.9, 0.99)), 640), LC.layer(LC.heads(1, 1, 64, 40, 64), LC.ret(16, 16, (0.9,)), None)], side=24, loop=(1, 2, 2))
    w = LC.weights(cfg, 32)
    m = LugasunForCausalLM.from_state_dict(w, cfg, dtype=dtype, max_tokens=64, max_seqs=20)
    toks = [LC.tokens(cfg, 12, seed=i) for i in range(20)]

    def run(which):
        for i in which:
            m.step([(i, toks[i][:9], [])])
        z = torch.stack([m.step([(i, [toks[i][9 + k]], [0]) for i in which]) for k in range(3)], 1).cpu()
        for i in which:
            m.end(i)
        return z
    together = run(range(20))
    assert LC.close(together[5], O.forward(w, cfg, toks[5])[9:], dtype)
    for which in ([0], [3], [0, 1], [4, 5, 6, 7], range(8)):
        assert torch.equal(run(which), together[list(which)]), which
    m.close()


@pytest.mark.parametrize('dim', [16, 64])
def test_decoded_state_steps_as_prompts_do(dim):
    """float32, states of up to 64 keys: a decoded token moves its state as a prompt's token does, decay times state rounded ahead of the fused k v.  With one live value column the outputs' norms are
    the same sums too, so decoded logits have the bits of the prompt that holds their tokens."""
    from callireader_amd.modeling_decoder import LugasunForCausalLM
    cfg = LC.config(128, 90, [LC.layer(LC.heads(1, 1, 64, 64, 64), LC.ret(dim, 16, (0.9, 0.97, 0.999)), None, (0.0, 0.8))], side=8)
    w = LC.weights(cfg, 43)
    v = w['l0.mix.right.v'].view(3, 16, 128)
    v[:, 1:] = 0
    m = LugasunForCausalLM.from_state_dict(w, cfg, dtype=torch.float32, max_tokens=64, max_seqs=2)
    t = LC.tokens(cfg, 60, seed=9)
    whole = m.step([('prompt', t, list(range(40, 60)))])
    m.step([('row', t[:40], [])])
    rows = torch.cat([m.step([('row', [x], [0])]) for x in t[40:]])
    torch.cuda.synchronize()
    assert torch.equal(rows, whole), float((rows - whole).abs().max())
    m.close()


@pytest.mark.parametrize('dtype', [F32, BF16])
@pytest.mark.parametrize('rows', [1, 3, 8])
@pytest.mark.parametrize('width,ff,ret_heads', [(1024, 640, 1), (1152, 1152, 3), (2048, 4096, 4)])
def test_weights_fetched_beside_a_mixer(width, ff, ret_heads, rows, dtype, monkeypatch):
    """Behind a mixer's own workgroups others read the next products' weights: counts of own workgroups that eight does and does not divide, products of tiles that eight does not divide, which are left
    out, the last layer of a span with the embedding's product next and the last of all with none.  The separate kernels fetch nothing: the same bits, for reading leaves nothing behind.  What is
    read is tests/test_l2_ahead_cpu.py's to say."""
    from callireader_amd.modeling_decoder import LugasunForCausalLM
    layer = LC.layer(LC.heads(2, 1, 64, 64, 64), LC.ret(64, 64, (0.97,) * ret_heads), ff)
    cfg = LC.config(width, 90, [layer, layer, LC.layer(LC.heads(1, 1, 64, 40, 64), LC.ret(16, 16, (0.9,)), None)], side=24, loop=(1, 2, 2))
    w = LC.weights(cfg, 35)
    toks = [LC.tokens(cfg, 12 + i, seed=i) for i in range(rows)]
    got = []
    for joined in ('1', '0'):
        monkeypatch.setenv('CR_DECODE_JOINED', joined)
        m = LugasunForCausalLM.from_state_dict(w, cfg, dtype=dtype, max_tokens=64, max_seqs=rows)
        for i, t in enumerate(toks):
            m.step([(i, t[:-3], [])])
        got.append(torch.stack([m.step([(i, [t[len(t) - 3 + k]], [0]) for i, t in enumerate(toks)]) for k in range(3)]).cpu())
        m.close()
    assert torch.isfinite(got[0]).all() and torch.equal(*got)
