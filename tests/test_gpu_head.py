"""The vocabulary head with the final norm in front, against the norm and the head as launches of their own (what a model whose decode
copies were dropped takes): the same bits, at row counts that leave wavefronts without a row, with 63 to 65 and with more than 64."""
import numpy as np
import pytest

import util
from cera_amd import hip_api, host_api as H, synth

pytestmark = pytest.mark.gpu


def _same_as_apart(hip, cfg, weights):
    m = hip_api.Model(hip, cfg, weights)
    fused = [m.forward(3, 0), m.forward_prefill([5, 1, 4], 1), m.read_hidden()]
    m.truncate_kv(0)
    m.drop_decode_copies()
    apart = [m.forward(3, 0), m.forward_prefill([5, 1, 4], 1), m.read_hidden()]
    m.close()
    for a, b in zip(fused, apart):
        assert np.isfinite(a).all() and np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.parametrize("hidden", [256, 2304, 4352])
@pytest.mark.parametrize("head", [H.Q4_K, H.Q6_K, H.Q4_0, H.Q4_1, H.Q8_0])
def test_head_types_and_row_lengths(hip, head, hidden):
    print(f"head type {head}, {hidden} columns", flush=True)
    cfg = {**synth.TINY, "hidden": hidden, "n_layers": 1, "vocab": 300}
    weights = synth.make_llama(cfg, seed=5, sigma=0.05, type_of=lambda n: H.Q4_K)
    weights["output.weight"] = (head, 300, hidden, util.make_weights(head, 300, hidden, 6, 0.05)[0])
    _same_as_apart(hip, cfg, weights)


@pytest.mark.parametrize("vocab", [6, 9, 4095, 4097, 12289, 262143, 262145, 270001])
def test_head_row_counts(hip, vocab):
    print(f"head of {vocab} rows", flush=True)
    cfg = dict(synth.TINY)
    weights = synth.make_llama(cfg, seed=78, sigma=0.05)
    for name in ("token_embd.weight", "output.weight"):
        t, rows, k, blocks = weights[name]
        weights[name] = (t, vocab, k, np.ascontiguousarray(np.resize(blocks.reshape(rows, -1), (vocab, blocks.size // rows))))
    _same_as_apart(hip, {**cfg, "vocab": vocab}, weights)
