"""One position's logits written by the head's launch into the model's pinned row: after prompts, steps and greedy steps in turn, with a
logit scale (whose launch behind the head takes the other route), and from two models of one context in two threads.  Bit for bit."""
import threading

import numpy as np
import pytest

import fidinex_util as F
import test_gpu_fidinex as TF
from cera_amd import hip_api, synth

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.ascontiguousarray(a).view(np.uint32)


@pytest.mark.parametrize("scale", [1.0, 4.0])
def test_steps_prompts_and_greedy_steps_in_turn(hip, scale):
    cfg = dict(synth.TINY)
    weights = synth.make_llama(cfg, seed=78, sigma=0.05)
    plain = hip_api.Model(hip, cfg, weights)
    m = hip_api.Model(hip, {**cfg, "logit_scale": scale}, weights)
    toks, kept = [3, 9, 1, 7, 2, 5], []
    for model in (plain, m):
        a = model.forward_prefill(toks[:4], 0)
        b = model.forward(toks[4], 4)
        nxt = model.forward_greedy(toks[5], 5)
        c = model.forward(nxt, 6)
        kept.append((a, b, c, nxt))
    want, got = kept
    assert got[3] == want[3]
    for x, y in zip(got[:3], want[:3]):
        assert np.array_equal(_bits(x), _bits(y * np.float32(1 / scale)))   # a power of two: exact
    again = [m.forward_prefill(toks[:4], 0), m.forward(toks[4], 4)]
    assert np.array_equal(_bits(again[0]), _bits(got[0])) and np.array_equal(_bits(again[1]), _bits(got[1]))
    m.close()
    plain.close()


def test_two_models_of_one_context_in_two_threads(hip, tmp_path):
    cfg = dict(synth.TINY)
    models = [hip_api.Model(hip, cfg, synth.make_llama(cfg, seed=s, sigma=0.05)) for s in (79, 80)]
    alone = [[m.forward(t, p) for p, t in enumerate((4, 8, 2, 6))] for m in models]
    both = [[], []]

    def run(i):
        for _ in range(10):
            both[i].append([models[i].forward(t, p) for p, t in enumerate((4, 8, 2, 6))])

    threads = [threading.Thread(target=run, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i in range(2):
        assert len(both[i]) == 10
        for seen in both[i]:
            assert all(np.array_equal(_bits(a), _bits(b)) for a, b in zip(seen, alone[i]))
        models[i].close()


@TF.DTYPES
def test_layered_steps_and_prompts(tmp_path, f32):
    cfg = F.config([F.attention(4, 2, 16, 16, (0.3, 8), True, ff=72)], width=84, vocab=1001, streams=4)
    w = F.random_model(cfg, 81)
    m = TF._open(F.save(tmp_path / "m", cfg, w), f32)
    toks = F.tokens(cfg, 12, 3)
    want = F.reference(cfg, w, toks)
    got = [m.forward_prefill(toks[:10], 0), m.forward(int(toks[10]), 10), m.forward(int(toks[11]), 11)]
    assert F.rel(np.stack(got), want[9:]) < TF.TOL[f32]
    m.close()
