"""What this framework's users have it do, as measurable cases: pictures into visual tokens, character tiles into pseudo-tokens, and language models of every design it runs from
prompt to answer.

  see     T tiles of 448 x 448 through the 24-layer vision tower and the projector: `InternVLChatModel.extract_feature` (a picture in a chat, the tiles of a page)
  align   T character tiles through the same and the resampler, then the cosine-VQ lookup and the de-normalisation of their pseudo-tokens: the steps of
          `InternVLChatModel.generate` ahead of its splice.  The lookup is given pseudo-tokens near rows of its table, as a trained resampler's are (a random one's
          have no nearest row that rounding would not change)
  answer  `rows` prompts prefilled together, then `new` steps in which every row is given its next token and its logits are read: InternLM2 layers through the model's engine
          (`prefill_batch`, `decode`), text models through `DecoderLM.step`, as generation and a replayed trace drive them; `new` = 0 only reads the prompts

Language models have the full width of their design and a few of its layers (every layer costs the same); the vision tower and the resampler are whole.  Weights are random, in the
checkpoint's shapes.  Decode steps are given their tokens, so that outputs can be compared: greedy picks of random weights hang on the last bit.
"""
import math

import torch
import torch.nn.functional as F

from callireader_amd import modeling_decoder, synthetic
from callireader_amd.config import DecoderSpec, ModelDims
from callireader_amd.modeling_internvl_chat import InternVLChatModel

CHAT_LAYERS, RESAMPLER_LAYERS = 4, 4


def _linasun(width, heads, dim, q_rank, kv_rank, experts, top, ff, groups, layers, vocab, loop=None):
    layer = dict(type='latent_attention', mixer=dict(heads=heads, dim=dim, vdim=dim, q_rank=q_rank, kv_rank=kv_rank, scale=dim ** -0.5),
                 mlp=dict(kind='moe', expert=dict(ff=ff, limit=7.0), router=dict(experts=experts, top=top, groups=dict(count=groups[0], keep=groups[1]))))
    return dict(architecture='Linasun', width=width, vocab=vocab, norm=dict(eps=1e-6), logit_softcap=30.0, layers=[layer] * layers,
                **({'loop': dict(start=loop[0], stop=loop[1], times=loop[2])} if loop else {}))


def _lugasun(width, heads, kv_heads, dim, chunk, ret_heads, ret_dim, ret_vdim, ff, side, layers, vocab, loop=None):
    left = dict(heads=heads, kv_heads=kv_heads, dim=dim, vdim=dim, mask=dict(size=chunk), scale=dim ** -0.5, softcap=50.0, rot=dict(base=1e6, dims=dim))
    right = dict(heads=ret_heads, dim=ret_dim, vdim=ret_vdim, decay=[1.0 - 2.0 ** (-5 - 6 * i / ret_heads) for i in range(ret_heads)], rot=dict(base=1e4, dims=ret_dim))
    layer = dict(type='parallel', mixer=dict(left=left, right=right, left_scale=0.7, right_scale=0.7), mlp=dict(kind='dense', ff=ff))
    return dict(architecture='Lugasun', width=width, vocab=vocab, norm=dict(eps=1e-6), layers=[layer] * layers, token_side=dict(dim=side),
                **({'loop': dict(start=loop[0], stop=loop[1], times=loop[2])} if loop else {}))


# the sizes `bench.py --workload linasun | lugasun` measures, but for the widest; one group of experts more is open, so that a group's last place is not a matter of rounding
TEXT = {
    'linasun_2048': _linasun(2048, 16, 128, 768, 512, 32, 4, 1024, (4, 3), 8, 32000),
    'linasun_looped': _linasun(1024, 8, 128, 384, 256, 16, 2, 1024, (4, 3), 6, 32000, loop=(1, 5, 3)),
    'lugasun_2048': _lugasun(2048, 16, 4, 128, 1024, 8, 128, 256, 8192, 128, 8, 32000),
    'lugasun_looped': _lugasun(1024, 8, 2, 128, 512, 8, 64, 64, 4096, 64, 6, 32000, loop=(1, 5, 3)),
}


def listed():
    chat = dict(kind='answer', model='internlm2', dtype='bfloat16')
    text = dict(kind='answer', dtype='bfloat16')
    return [
        # one picture of at most one tile shown in a chat: the smallest visual call
        dict(name='picture', kind='see', tiles=1),
        # the tiles of a 788 x 2000 page: 2 x 5 and its thumbnail
        dict(name='page', kind='see', tiles=11),
        # the characters that the detector finds on that page
        dict(name='characters', kind='align', tiles=96),
        # a question without a picture, answered alone
        dict(chat, name='question', rows=1, prompt=77, new=16),
        # the answer to one page: its visual and pseudo-tokens and the question are 3164 positions
        dict(chat, name='page_answer', rows=1, prompt=3164, new=32),
        # a GPU's share of 64 pages spread over the ranks that own them
        dict(chat, name='pages_13', rows=13, prompt=3164, new=24),
        # as many short requests as a decode batch holds
        dict(chat, name='requests_64', rows=64, prompt=333, new=24),
        # text models: documents read (an odd length), a batch of short requests, one request alone, portions of a document longer than a chunk, and 32-bit arithmetic
        dict(text, name='latent_documents', model='linasun_2048', rows=4, prompt=1531, new=0),
        dict(text, name='latent_requests', model='linasun_2048', rows=24, prompt=64, new=32),
        dict(text, name='retention_documents', model='lugasun_2048', rows=4, prompt=2048, new=4),
        dict(text, name='retention_request', model='lugasun_looped', rows=1, prompt=48, new=32),
        dict(text, name='retention_fp32', model='lugasun_looped', rows=2, prompt=201, new=12, dtype='float32'),
    ]


def _between(rng, lo, hi):
    """A whole number whose logarithm is uniform."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(['see', 'align', 'chat', 'chat', 'text', 'text', 'text32'])
    if kind in ('see', 'align'):
        return dict(kind=kind, tiles=_between(rng, 1, 40 if kind == 'see' else 96))
    if kind == 'chat':
        rows, prompt = _between(rng, 1, 64), _between(rng, 20, 3300)
        return dict(kind='answer', model='internlm2', dtype='bfloat16', rows=rows, prompt=max(20, min(prompt, 32768 // rows)), new=rng.randint(2, 24))
    model = rng.choice(sorted(TEXT))
    if kind == 'text32':
        return dict(kind='answer', model=rng.choice(['linasun_looped', 'lugasun_looped']), dtype='float32', rows=rng.randint(1, 8), prompt=_between(rng, 12, 200), new=rng.randint(1, 12))
    rows, prompt = _between(rng, 1, 64), _between(rng, 12, 3000)
    return dict(kind='answer', model=model, dtype='bfloat16', rows=rows, prompt=max(12, min(prompt, 8192 // rows)), new=rng.randint(0, 32))


# ---- inputs ----------------------------------------------------------------------------------------
DEV = 'cuda'


def _gen(seed, what):
    return torch.Generator(device=DEV).manual_seed((seed * 1000003 + what) % (1 << 62))


def _dims(c):
    if c['kind'] == 'see':
        return ModelDims.reduced(vit_layers=24, rs_depth=0, llm_layers=0), ('vit', 'mlp1')
    if c['kind'] == 'align':
        return ModelDims.reduced(vit_layers=24, rs_depth=RESAMPLER_LAYERS, llm_layers=0), ('vit', 'mlp1', 'resampler', 'vq')
    return ModelDims.reduced(vit_layers=0, rs_depth=0, llm_layers=CHAT_LAYERS), ('llm',)


def _weights(c, seed):
    """(checkpoint name, bf16 tensor), drawn on the GPU one by one."""
    g = _gen(seed, 1)
    if c['kind'] != 'answer' or c['model'] == 'internlm2':
        dims, parts = _dims(c)
        for name, (shape, std, mean) in synthetic.key_specs(dims, parts).items():
            if name.endswith(('wo.weight', 'w2.weight')):
                std /= 8                                                                  # what a layer adds is small beside the stream, as in a trained model
            if name.endswith('tok_embeddings.weight'):
                std = 0.5
            yield name, torch.empty(shape, device=DEV).normal_(mean, std, generator=g).to(torch.bfloat16)
        return
    spec = _spec(c)
    for name, shape in spec.weight_shapes().items():
        leaf = name.rsplit('.', 1)[-1]
        r = torch.randn(*shape, device=DEV, generator=g)
        if len(shape) == 1:
            r = 0.1 * r - 0.85 if leaf in ('norm1b', 'norm2b') else 1.0 + 0.1 * r if spec.norm_plain or (leaf == 'norm' and name != 'final.norm') else (1e-6 if leaf == 'correction' else 0.1) * r
        elif name != 'embed':
            r = r * ((6.0 if leaf == 'router' else 1.0) / math.sqrt(shape[1]))            # (a router that has made up its mind: with flat scores the choice is rounding)
        yield name, r.to(torch.bfloat16)


def _spec(c):
    cfg = TEXT[c['model']]
    return (DecoderSpec.from_linasun if cfg['architecture'] == 'Linasun' else DecoderSpec.from_lugasun)(cfg)


def _pixels(c, seed):
    return torch.empty(c['tiles'], 3, 448, 448, device=DEV).normal_(generator=_gen(seed, 2)).to(torch.bfloat16)      # (ImageNet-normalised pixels)


def _embeds(c, seed):
    """Prompt embeddings, as a splice leaves them: [rows, prompt, width]."""
    return (0.5 * torch.randn(c['rows'], c['prompt'], 4096, device=DEV, generator=_gen(seed, 3))).to(torch.bfloat16)


def _tokens(c, seed, vocab):
    """[rows, prompt + new] token ids, on the host."""
    return torch.randint(0, vocab, (c['rows'], c['prompt'] + c['new']), generator=torch.Generator().manual_seed(seed * 7919 + 4))


def _pseudo(c, seed, table):
    """Pseudo-tokens as a trained resampler gives them, near rows of the table: [tiles, 3, width]."""
    g = _gen(seed, 5)
    at = torch.randint(0, len(table), (c['tiles'], 3), device=DEV, generator=g)
    return (table[at].float() + 0.5 * torch.randn(c['tiles'], 3, table.shape[1], device=DEV, generator=g)).to(torch.bfloat16)


def prepare(c, seed):
    if c['kind'] != 'answer':
        dims, _ = _dims(c)
        w = dict(_weights(c, seed))
        pseudo = _pseudo(c, seed, w['normed_emb.weight']) if c['kind'] == 'align' else None
        return dict(case=c, model=InternVLChatModel.from_state_dict(w, dims, max_tokens=64), pixels=_pixels(c, seed), pseudo=pseudo)
    room = c['prompt'] + c['new'] + 1
    if c['model'] == 'internlm2':
        dims, _ = _dims(c)
        m = InternVLChatModel.from_state_dict(_weights(c, seed), dims, max_tokens=room)
        given = _tokens(c, seed, dims.vocab)[:, c['prompt']:].to(DEV)
        return dict(case=c, model=m, kv=m.engine.kv_alloc(c['rows'], room), embeds=list(_embeds(c, seed)), given=[given[:, t].contiguous() for t in range(c['new'])])
    cls = modeling_decoder.LinasunForCausalLM if 'linasun' in c['model'] else modeling_decoder.LugasunForCausalLM
    m = cls.from_state_dict(_weights(c, seed), _spec(c), dtype=getattr(torch, c['dtype']), max_tokens=room, max_seqs=c['rows'])
    toks = _tokens(c, seed, m.spec.vocab).tolist()
    n = c['prompt']
    return dict(case=c, model=m, prompts=[(i, t[:n], [n - 1]) for i, t in enumerate(toks)], given=[[(i, [t[n + s]], [0]) for i, t in enumerate(toks)] for s in range(c['new'])])


# ---- one pass --------------------------------------------------------------------------------------
def run(s):
    c, m = s['case'], s['model']
    with torch.inference_mode():
        if c['kind'] == 'see':
            return m.extract_feature(s['pixels'])
        if c['kind'] == 'align':
            feats = m.extract_feature(s['pixels'])
            out = m.resampler(feats)
            idx = m.engine.vq(s['pseudo'])
            return feats, out, idx, m.engine.denorm(s['pseudo'], idx)
        if c['model'] == 'internlm2':
            e, kv, rows = m.engine, s['kv'], list(range(c['rows']))
            kv.reset()
            logits = [e.prefill_batch(kv, rows, s['embeds'], want_logits=True)]
            for t in s['given']:
                logits.append(e.decode(kv, rows, force_tokens=t, want_logits=True))
            return logits
        logits = [m.step(s['prompts'])]
        for entries in s['given']:
            logits.append(m.step(entries))
        for rid, _, _ in s['prompts']:
            m.end(rid)
        return logits


# ---- what a pass cannot do without -----------------------------------------------------------------
def work(c):
    if c['kind'] != 'answer':
        T = c['tiles']
        w = 304e6 + 33.6e6                                                             # vision tower and projector weights
        flops, byts = T * (723.6e9 + 17.18e9), 2 * (w + T * (3 * 448 * 448 + 256 * 4096))
        if c['kind'] == 'align':
            flops += T * (12.02e9 + 2.27e9)
            byts += 2 * (569e6 + 92553 * 4096 + T * (256 * 4096 + 6 * 4096)) + T * 3 * 8
        return dict(bytes=byts, flops=flops)
    R, S, N = c['rows'], c['prompt'], c['new']
    es = 4 if c['dtype'] == 'float32' else 2
    if c['model'] == 'internlm2':
        lin, head, L = 4096 * 6144 + 4096 * 4096 + 3 * 4096 * 14336, 4096 * 92553, CHAT_LAYERS
        flops = 2.0 * R * (S * lin * L + head + S * (S + 1) / 2 * 2 * 4096 * L) + 2.0 * R * N * (lin * L + head + (S + N / 2) * 2 * 4096 * L)
        kv = 2 * 2 * 8 * 128 * L
        byts = (N + 1) * (2.0 * (lin * L + head) + 4.0 * R * 92553) + R * (2 * 4096 * S + kv * (S + N) + kv * N * (S + N / 2))
        return dict(bytes=byts, flops=flops)
    spec = _spec(c)
    V, W = spec.vocab, spec.width
    cfg = TEXT[c['model']]['layers'][0]
    P = len(spec.passes)
    if 'linasun' in c['model']:
        m, r, e = cfg['mixer'], cfg['mlp']['router'], cfg['mlp']['expert']
        mix = W * (m['q_rank'] + m['kv_rank'] + 2 * m['heads'] * m['vdim']) + m['q_rank'] * m['heads'] * m['dim'] + m['kv_rank'] * m['heads'] * (m['dim'] + m['vdim'])
        one, active = 3 * W * e['ff'], mix + W * r['experts'] + r['top'] * 3 * W * e['ff']
        read = lambda n: mix + W * r['experts'] + r['experts'] * (1 - (1 - r['top'] / r['experts']) ** n) * one      # noqa: E731  (experts that n tokens are expected to choose)
        keys, cache, state = m['heads'] * (m['dim'] + m['vdim']), m['kv_rank'], 0
        sees = lambda n: n * (n + 1) / 2                                               # noqa: E731
        extra = 0
    else:
        a, t = cfg['mixer']['left'], cfg['mixer']['right']
        active = W * (a['heads'] + a['kv_heads']) * 2 * a['dim'] + W * t['heads'] * (2 * t['dim'] + 3 * t['vdim']) + 2 * W * cfg['mlp']['ff'] + 2 * W * TEXT[c['model']]['token_side']['dim']
        read = lambda n: active                                                        # noqa: E731
        keys, cache, state = a['heads'] * 2 * a['dim'], a['kv_heads'] * 2 * a['dim'], t['heads'] * t['dim'] * t['vdim']
        ch = a['mask']['size']
        sees = lambda n: n // ch * ch * (ch + 1) / 2 + (n % ch) * (n % ch + 1) / 2     # noqa: E731
        extra = (spec.loop[2] if spec.loop else 0) * 2 * W * W
    flops = 2.0 * R * (S + N) * (P * (active + 2 * state) + extra) + 2.0 * R * sees(S + N) * keys * P + 2.0 * R * (N + 1) * W * V
    seen = (sees(S + N) - sees(S)) if N else 0                                          # keys that the decode steps read
    byts = es * (P * read(R * S) + extra + W * V) + N * es * (P * read(R) + extra + W * V) + 4.0 * R * (N + 1) * V + R * P * (es * cache * (S + N + seen) + 4 * state * (1 + 2 * N))
    return dict(bytes=byts, flops=flops)


def tolerance(c):
    return dict(rel=5e-5) if c.get('dtype') == 'float32' else dict(rel=3e-2)


# ---- the same in 64 bits ---------------------------------------------------------------------------
def _lin(x, w, b=None):
    y = x @ w.double().T
    return y if b is None else y + b.double()


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _ln(x, w, b, eps):
    return F.layer_norm(x, x.shape[-1:], w.double(), b.double(), eps)


def _rotate(x, base, dims):
    """x [tokens, heads, dim]: entries i and i + dims / 2 turn by position * base^(-2 i / dims)."""
    half = dims // 2
    a = torch.arange(x.shape[0], device=x.device, dtype=torch.float64)[:, None] * base ** (-2.0 * torch.arange(half, device=x.device, dtype=torch.float64) / dims)
    cos, sin = a.cos()[:, None], a.sin()[:, None]
    u, v = x[..., :half], x[..., half:dims]
    return torch.cat([u * cos - v * sin, v * cos + u * sin, x[..., dims:]], -1)


def _attend(q, k, v, scale, cap=None, chunk=None):
    """q [n, H, d], k / v [n, G, d] -> [n, H, d], causal, head by head."""
    n, H, G = q.shape[0], q.shape[1], k.shape[1]
    i = torch.arange(n, device=q.device)
    hidden = i[None] > i[:, None]
    if chunk:
        hidden |= i[None] // chunk != i[:, None] // chunk
    out = torch.empty(n, H, v.shape[2], device=q.device, dtype=torch.float64)
    for h in range(H):
        s = q[:, h] @ k[:, h * G // H].T.contiguous() * scale
        if cap:
            s = cap * torch.tanh(s / cap)
        out[:, h] = torch.softmax(s.masked_fill_(hidden, -math.inf), -1) @ v[:, h * G // H].contiguous()
    return out


def _each(rows, n, f, *xs):
    """f on every row's n tokens of tensors [rows * n, ...]."""
    return torch.cat([f(*(x[r * n:(r + 1) * n] for x in xs)) for r in range(rows)])


def _see64(w, px):
    x = F.unfold(px.double(), 14, stride=14).transpose(1, 2)
    v = 'vision_model.embeddings.'
    x = _lin(x, w[v + 'patch_embedding.weight'].flatten(1), w[v + 'patch_embedding.bias'])
    x = torch.cat([w[v + 'class_embedding'].double().expand(len(x), 1, -1), x], 1) + w[v + 'position_embedding'].double()
    for i in range(24):
        p = f'vision_model.encoder.layers.{i}.'
        h = _ln(x, w[p + 'norm1.weight'], w[p + 'norm1.bias'], 1e-6)
        q, k, u = (t.contiguous() for t in _lin(h, w[p + 'attn.qkv.weight'], w[p + 'attn.qkv.bias']).view(len(x), 1025, 3, 16, 64).permute(2, 0, 3, 1, 4))
        a = (torch.softmax(q * 0.125 @ k.transpose(-1, -2).contiguous(), -1) @ u).transpose(1, 2).reshape(x.shape)
        x = x + _lin(a, w[p + 'attn.proj.weight'], w[p + 'attn.proj.bias']) * w[p + 'ls1'].double()
        h = F.gelu(_lin(_ln(x, w[p + 'norm2.weight'], w[p + 'norm2.bias'], 1e-6), w[p + 'mlp.fc1.weight'], w[p + 'mlp.fc1.bias']))
        x = x + _lin(h, w[p + 'mlp.fc2.weight'], w[p + 'mlp.fc2.bias']) * w[p + 'ls2'].double()
    # 2 x 2 neighbours into one token, in the checkpoint's order: the two columns of a row side by side, one such row after the other, twice
    x = x[:, 1:].reshape(len(x), 32, 16, 2048).permute(0, 2, 1, 3).reshape(len(x), 16, 16, 4096).permute(0, 2, 1, 3).reshape(len(x), 256, 4096)
    h = F.gelu(_lin(_ln(x, w['mlp1.0.weight'], w['mlp1.0.bias'], 1e-5), w['mlp1.1.weight'], w['mlp1.1.bias']))
    return _lin(h, w['mlp1.3.weight'], w['mlp1.3.bias'])


def _resample64(w, x):
    y = w['resampler.learns'].double().expand(len(x), 3, -1)
    split = lambda t: t.reshape(len(x), -1, 8, 64).transpose(1, 2).contiguous()          # noqa: E731
    for i in range(RESAMPLER_LAYERS):
        p, f = f'resampler.layers.{i}.0.', f'resampler.layers.{i}.1.net.'
        m, z = _ln(x, w[p + 'norm_media.weight'], w[p + 'norm_media.bias'], 1e-5), _ln(y, w[p + 'norm_learns.weight'], w[p + 'norm_learns.bias'], 1e-5)
        k, v = _lin(torch.cat([m, z], 1), w[p + 'to_kv.weight']).chunk(2, -1)
        a = torch.softmax(split(_lin(z, w[p + 'to_q.weight'])) * 0.125 @ split(k).transpose(-1, -2).contiguous(), -1) @ split(v)
        y = y + _lin(a.transpose(1, 2).reshape(len(x), 3, 512), w[p + 'to_out.weight'])
        h = F.gelu(_lin(_ln(y, w[f + '0.weight'], w[f + '0.bias'], 1e-5), w[f + '1.weight'], w[f + '1.bias']))
        y = y + _lin(h, w[f + '3.weight'], w[f + '3.bias'])
    return _ln(y, w['resampler.norm.weight'], w['resampler.norm.bias'], 1e-5)


def _internlm64(w, x, rows):
    n = len(x) // rows
    for i in range(CHAT_LAYERS):
        p = f'language_model.model.layers.{i}.'
        qkv = _lin(_rms(x, 1e-5) * w[p + 'attention_norm.weight'].double(), w[p + 'attention.wqkv.weight']).view(-1, 8, 6, 128)

        def heads(t):
            return _attend(_rotate(t[:, :, :4].reshape(n, 32, 128), 1e6, 128), _rotate(t[:, :, 4], 1e6, 128), t[:, :, 5], 128 ** -0.5).reshape(n, 4096)
        x = x + _lin(_each(rows, n, heads, qkv), w[p + 'attention.wo.weight'])
        h = _rms(x, 1e-5) * w[p + 'ffn_norm.weight'].double()
        x = x + _lin(F.silu(_lin(h, w[p + 'feed_forward.w1.weight'])) * _lin(h, w[p + 'feed_forward.w3.weight']), w[p + 'feed_forward.w2.weight'])
    return _rms(x, 1e-5) * w['language_model.model.norm.weight'].double()


def _linasun64(w, cfg, spec, tok, rows):
    n, W, eps = len(tok) // rows, cfg['width'], cfg['norm']['eps']
    norm = lambda x, g: _rms(x, eps) * (1.0 + w[g].double())                             # noqa: E731
    j = torch.arange(W, device=tok.device)
    a = torch.arange(n, device=tok.device).double()[:, None] * 10000.0 ** (-2.0 * (j // 2).double() / W)
    x = w['embed'].double()[tok] + torch.where(j % 2 == 0, a.sin(), a.cos()).repeat(rows, 1)
    for i in spec.passes:
        s, p, f = cfg['layers'][i]['mixer'], f'l{i}.mix.', f'l{i}.mlp.'
        h = norm(x, f'l{i}.norm1')
        c = _rms(_lin(h, w[p + 'dkv']), eps) * w[p + 'dkv.norm'].double()
        q = _lin(_rms(_lin(h, w[p + 'dq']), eps) * w[p + 'dq.norm'].double(), w[p + 'uq'])
        o = _each(rows, n, lambda *t: _attend(*(u.view(n, s['heads'], -1) for u in t), s['scale']).reshape(n, -1), q, _lin(c, w[p + 'uk']), _lin(c, w[p + 'uv']))
        x = x + norm(_lin(o * torch.sigmoid(_lin(h, w[p + 'g'])), w[p + 'o']), f'l{i}.norm1b')
        h, m = norm(x, f'l{i}.norm2'), cfg['layers'][i]['mlp']
        r = m['router']
        score = torch.softmax(_lin(h, w[f + 'router']), -1)
        pick = (score + w[f + 'correction'].double()).view(len(x), r['groups']['count'], -1)
        shut = torch.ones(pick.shape[:2], dtype=torch.bool, device=x.device).scatter_(1, pick.max(-1).values.topk(r['groups']['keep'], -1).indices, False)
        idx = pick.masked_fill(shut[:, :, None], -math.inf).flatten(1).topk(r['top'], -1).indices
        y = torch.zeros_like(x)
        for e in range(r['experts']):
            at, slot = (idx == e).nonzero(as_tuple=True)
            g, u = _lin(h[at], w[f'{f}e{e}.gate']).clamp(max=m['expert']['limit']), _lin(h[at], w[f'{f}e{e}.up']).clamp(-m['expert']['limit'], m['expert']['limit'])
            y[at] += score[at, e, None] * _lin(g * torch.sigmoid(1.702 * g) * (u + 1.0), w[f'{f}e{e}.down'])
        x = x + norm(y, f'l{i}.norm2b')
    return norm(x, 'final.norm')


def _lugasun64(w, cfg, spec, tok, rows):
    n, eps, D = len(tok) // rows, cfg['norm']['eps'], cfg['token_side']['dim']
    norm = lambda x, g: _rms(x, eps) * w[g].double()                                     # noqa: E731
    x0 = x = w['embed'].double()[tok]
    loop = cfg.get('loop')
    behind = torch.arange(n, device=tok.device, dtype=torch.float64)
    behind = behind[:, None] - behind[None]
    for at, i in enumerate(spec.passes):
        if loop and i == loop['start'] and at >= loop['start']:
            x = _lin(torch.cat([x, x0], -1), w['loop.in'])
        s, p = cfg['layers'][i]['mixer'], f'l{i}.mix.'
        a, t = s['left'], s['right']
        h = norm(x, f'l{i}.norm1')

        def left(q, k, v):
            q, k = (_rotate(_rms(u.view(n, -1, a['dim']), eps) * w[f'{p}left.{g}.norm'].double(), a['rot']['base'], a['rot']['dims']) for u, g in ((q, 'q'), (k, 'k')))
            return _attend(q, k, v.view(n, -1, a['vdim']), a['scale'], a['softcap'], a['mask']['size']).reshape(n, -1)

        def right(q, k, v):
            q, k, v = _rotate(q.view(n, t['heads'], -1), t['rot']['base'], t['rot']['dims']), _rotate(k.view(n, t['heads'], -1), t['rot']['base'], t['rot']['dims']), v.view(n, t['heads'], -1)
            out = []
            for b in range(t['heads']):
                fade = torch.where(behind >= 0, t['decay'][b] ** behind.clamp(min=0), 0.0)
                out.append(_rms((q[:, b] @ k[:, b].T.contiguous() * t['dim'] ** -0.5 * fade) @ v[:, b].contiguous(), eps))
            return torch.stack(out, 1).reshape(n, -1)
        l, r = (_each(rows, n, f, *(_lin(h, w[f'{p}{side}.{g}']) for g in 'qkv')) for f, side in ((left, 'left'), (right, 'right')))
        x = x + s['left_scale'] * _lin(l, w[p + 'left.o']) + s['right_scale'] * _lin(r * F.silu(_lin(h, w[p + 'right.g'])), w[p + 'right.o'])
        x = x + _lin(_lin(norm(x, f'l{i}.norm2'), w[f'l{i}.mlp.up']).relu().square(), w[f'l{i}.mlp.down'])
        e = w['side.embed'].double()[tok][:, i * D:(i + 1) * D]
        x = x + norm(_lin(F.gelu(_lin(x, w[f'l{i}.side.gate']), approximate='tanh') * e, w[f'l{i}.side.proj']), f'l{i}.side.norm')
    return norm(x, 'final.norm')


def exact(c, seed):
    with torch.inference_mode():
        w = dict(_weights(c, seed))
        if c['kind'] != 'answer':
            feats = torch.cat([_see64(w, px) for px in _pixels(c, seed).split(8)])
            if c['kind'] == 'see':
                return feats
            x, table = _pseudo(c, seed, w['normed_emb.weight']).double(), w['normed_emb.weight'].double()
            idx = (x.flatten(0, 1) @ F.normalize(table, dim=1).T.contiguous()).argmax(1)
            back = x.flatten(0, 1) * w['calli.sigma'].double()[idx] + w['calli.mu'].double()[idx]
            return feats, torch.cat([_resample64(w, f) for f in feats.split(16)]), idx.view(-1, 3), back
        R, S, N = c['rows'], c['prompt'], c['new']
        if c['model'] == 'internlm2':
            given = _tokens(c, seed, ModelDims.full().vocab)[:, S:].to(DEV)
            x = torch.cat([_embeds(c, seed).double(), w['language_model.model.tok_embeddings.weight'].double()[given]], 1).flatten(0, 1)
            x, head, cap = _internlm64(w, x, R), w['language_model.output.weight'], None
        else:
            cfg, spec = TEXT[c['model']], _spec(c)
            x = (_linasun64 if 'linasun' in c['model'] else _lugasun64)(w, cfg, spec, _tokens(c, seed, spec.vocab).to(DEV).flatten(), R)
            head, cap = w['embed' if spec.tied_head else 'head'], cfg.get('logit_softcap')
        x = x.view(R, S + N, -1)[:, S - 1:]
        z = [_lin(x[:, t].contiguous(), head) for t in range(N + 1)]
        return [cap * torch.tanh(v / cap) for v in z] if cap else z
