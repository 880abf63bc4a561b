"""Calls of one described decoder from several streams: each is ordered behind the last, whose workspace, cache and states it uses."""
import pytest
import torch

import lugasun_cases as LC
from callireader_amd.modeling_decoder import DecoderLM


def test_every_call_waits_for_the_stream_of_the_last(monkeypatch):
    log = []

    class Stream:
        def __init__(self, name):
            self.name = name

        def wait_stream(self, other):
            if other.name == 'gone':
                raise RuntimeError('no such stream')
            log.append((self.name, other.name))
    a, b = Stream('a'), Stream('b')

    class Calls:                                              # engine and slots in one: whatever is called is noted
        kv, slot = None, {'r': 0}

        def decode(self, *args, **kw):
            log.append('decode')
            return torch.zeros(1, 4)

        def prefill_tokens(self, *args, **kw):
            log.append('prefill')

        def release(self, rid):
            log.append('release')
    m = DecoderLM.__new__(DecoderLM)
    m.engine = m.slots = Calls()
    at = [a]
    monkeypatch.setattr(torch.cuda, 'current_stream', lambda *_: at[0])
    monkeypatch.setattr(torch.cuda, 'synchronize', lambda *_: log.append('synchronize'))
    m.step([('r', [1, 2], [])])
    m.step([('r', [3], [0])])
    at[0] = b
    m.step([('r', [4], [0])])
    m.step([('r', [5], [0])])
    at[0] = a
    m.end('r')
    assert log == ['prefill', 'decode', ('b', 'a'), 'decode', 'decode', ('a', 'b'), 'release']
    a.name = 'gone'                                           # a foreign stream that its owner has destroyed
    at[0] = b
    m.end('r')
    assert log[-2:] == ['synchronize', 'release']


@pytest.mark.gpu
@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
def test_steps_on_alternating_streams(dtype):
    """The same logits as on one stream, with work ahead of each step that holds its stream back."""
    from callireader_amd.modeling_decoder import LugasunForCausalLM
    cfg = LC.config(512, 90, [LC.layer(LC.heads(2, 1, 64, 64, 64), LC.ret(64, 64, (0.9, 0.99)), 640)] * 2, side=24)
    m = LugasunForCausalLM.from_state_dict(LC.weights(cfg, 61), cfg, dtype=dtype, max_tokens=64, max_seqs=2)
    t = [LC.tokens(cfg, 30, seed=i) for i in range(2)]

    def run(streams):
        z = []
        for k in range(20):
            s = streams[k % len(streams)]
            with torch.cuda.stream(s):
                if len(streams) > 1:
                    torch.cuda._sleep(200000 * (1 + k % 2))
                z.append(m.step([(i, t[i][:11] if k == 0 else [t[i][10 + k]], [0]) for i in range(2)]))
        torch.cuda.synchronize()
        for i in range(2):
            m.end(i)
        return torch.stack(z).cpu()
    one = run([torch.cuda.current_stream()])
    assert torch.equal(run([torch.cuda.Stream(), torch.cuda.Stream(), torch.cuda.current_stream()]), one)
    m.close()
