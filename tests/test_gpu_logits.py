"""What a step returns beside its pick: the head writes the caller's buffer itself where that is aligned to 16 bytes and no penalty is asked for, and fills a workspace that is
copied otherwise; rows asked for that are the last rows serve the pick too.  Both ways give the same bits, and the same next ids."""
import pytest
import torch

import linasun_cases as LC

pytestmark = pytest.mark.gpu


@pytest.fixture(params=['prompt embeddings', 'token ids'])
def engine(request):
    """(run, vocab): run(logits buffers of both calls' rows or None, penalty) -> the ids of three sequences after a prefill and a decode step"""
    import ctypes as C
    from callireader_amd import _binding as B
    if request.param == 'token ids':
        from callireader_amd.modeling_decoder import LinasunForCausalLM
        cfg = dict(LC.TINY, vocab=1003)
        m = LinasunForCausalLM.from_state_dict(LC.weights(cfg, 6), cfg, dtype=torch.float32, max_tokens=64, max_seqs=3)
        eng, vocab = m.engine, cfg['vocab']
    else:
        from callireader_amd import synthetic
        from callireader_amd.config import ModelDims
        from callireader_amd.engine import Engine
        dims = ModelDims.reduced(vit_layers=1, llm_layers=1, rs_depth=1, vocab=8201)
        eng, vocab, m = Engine(dims, max_pos=512), dims.vocab, None
        eng.load_state_dict(synthetic.make_state_dict(dims, parts=('llm',), seed=0))
        eng.load_rope()
        eng.finalize()
    kv = eng.kv_alloc(3, 64)
    lens, g = [5, 1, 20], torch.Generator().manual_seed(8)
    prompts = torch.cat([torch.randn(n, 4096, generator=g) * 0.02 for n in lens]).to('cuda', torch.bfloat16)
    flat = [t for n in lens for t in LC.tokens(dict(vocab=vocab), n, seed=n)]
    arr = lambda v, t=C.c_int32: (t * len(v))(*v)

    def run(last, step, penalty, want=None, asked=None):
        s, p = torch.cuda.current_stream().cuda_stream, lambda t: C.c_void_p(0 if t is None else t.data_ptr())
        kv.reset()
        if m is None:
            B.check(B.lib.cr_llm_prefill_batch(eng._h, kv._h, arr([2, 0, 1]), 3, p(prompts), arr(lens), penalty, p(last), s), 'prefill')
        else:
            B.check(B.lib.cr_llm_prefill_tokens(eng._h, kv._h, arr([2, 0, 1]), 3, arr(flat, C.c_int64), arr(lens), penalty, p(last), arr(want or [0]), len(want or []), p(asked), s), 'prefill')
        B.check(B.lib.cr_llm_decode(eng._h, kv._h, arr([2, 0, 1]), 3, C.c_void_p(0), penalty, p(step), s), 'decode')
        torch.cuda.synchronize()
        return [kv.generated(i) for i in range(3)]

    yield run, vocab, m is not None
    kv.free()
    if m is not None:
        m.close()


@pytest.mark.parametrize('penalty', [1.0, 1.3])
def test_logits_in_place_and_copied(engine, penalty):
    run, V, tokens = engine
    buf = lambda off: torch.full((3 * V + 4,), float('nan'), device='cuda')[off:off + 3 * V]
    ids = run(None, None, penalty)
    a, b = (buf(0), buf(0)), (buf(1), buf(3))                  # aligned | 4 and 12 bytes off
    assert run(*a, penalty) == ids and run(*b, penalty) == ids
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1]) and torch.isfinite(a[0]).all() and torch.isfinite(a[1]).all()
    if tokens:
        for want in ([4, 5, 25], [25, 0, 4]):                  # the last rows | others
            for off in (0, 1):
                last, asked = buf(off), buf(off)
                assert run(last, None, penalty, want, asked) == ids
                assert torch.equal(last, a[0])
                if want[0] == 4:
                    assert torch.equal(asked, a[0])
                else:
                    assert torch.equal(asked[:V], last[2 * V:]) and torch.equal(asked[2 * V:], last[:V])


@pytest.mark.parametrize('n', [1, 63, 64, 65, 255, 256])
def test_decode_attention_of_one_split(n):
    """A cache of at most 256 keys is one split, written by the kernel itself; counted as two splits, the second is empty and the combine kernel writes the row: the same bits."""
    from callireader_amd import engine as E
    g = torch.Generator().manual_seed(n)
    rand = lambda *s: torch.randn(*s, generator=g).to('cuda', torch.bfloat16)
    q, kc, vc = rand(3, 4096), rand(4, 8, 320, 128), rand(4, 8, 320, 128)
    seqs = torch.tensor([3, 0, 2], dtype=torch.int32, device='cuda')
    lens = torch.tensor([n - 1, 0, max(n - 2, 0), n // 2], dtype=torch.int32, device='cuda')
    one, two = (E.op_decode_attention(q, kc, vc, seqs, lens, max_keys=k) for k in (256, 257))
    assert torch.isfinite(one.float()).all() and torch.equal(one, two)


def test_rows_asked_for_in_a_long_call():
    """A call of more than 8190 prompt rows (its upload is past the heap's largest block), one row asked for of each prompt: the last ones, the ones ahead of them, the last ones in
    another order.  The picked ids are those of the last rows each time."""
    from callireader_amd.modeling_decoder import LinasunForCausalLM
    cfg = dict(LC.TINY, vocab=211)
    m = LinasunForCausalLM.from_state_dict(LC.weights(cfg, 6), cfg, dtype=torch.float32, max_tokens=2100, max_seqs=4)
    toks = [LC.tokens(cfg, 2050 - i, seed=i) for i in range(4)]

    def ids_and_logits(places):
        z = m.step([(i, t, [p]) for i, (t, p) in enumerate(zip(toks, places))])
        ids = [m.slots.kv.generated(m.slots.slot[i]) for i in range(4)]
        m.slots.clear()
        return ids, z

    last = [len(t) - 1 for t in toks]
    ids, z = ids_and_logits(last)
    assert ids == [[int(i)] for i in z.argmax(-1)] and torch.isfinite(z).all()
    other, z2 = ids_and_logits([p - 1 for p in last])
    assert other == ids and not torch.equal(z2, z)
    mixed, z3 = ids_and_logits(last[:2] + [0, 0])
    assert mixed == ids and torch.equal(z3[:2], z[:2])
    m.close()
