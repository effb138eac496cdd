"""Logits on their way to host memory: row counts around a whole 16-byte piece and around the pinned chunk.  A head of repeated rows
gives repeated logits, bit for bit, whichever route they take."""
import numpy as np
import pytest

from cera_amd import hip_api, synth

pytestmark = pytest.mark.gpu
CHUNK = 1 << 20


def _rows(weight, m):
    t, rows, k, blocks = weight
    return (t, m, k, np.ascontiguousarray(np.resize(blocks.reshape(rows, -1), (m, blocks.size // rows))))


@pytest.fixture(scope="module")
def base(hip):
    cfg = dict(synth.TINY)
    weights = synth.make_llama(cfg, seed=77, sigma=0.05)
    m = hip_api.Model(hip, cfg, weights)
    one, many = m.forward(3, 0), m.forward_prefill_logits_all([5, 1, 4], 1)
    m.close()
    return cfg, weights, one, many


ROWS = [6, 8, 513, 1000, CHUNK // 12, CHUNK // 12 + 1, CHUNK // 4, CHUNK // 4 + 4]


@pytest.mark.parametrize("vocab", ROWS)
def test_logits_of_any_number_of_rows(hip, base, vocab):
    cfg, weights, one, many = base
    print(f"logits to host: {vocab} rows", flush=True)
    w = {**weights, **{name: _rows(weights[name], vocab) for name in ("token_embd.weight", "output.weight")}}
    m = hip_api.Model(hip, {**cfg, "vocab": vocab}, w)
    got_one = m.forward(3, 0)
    got_many = m.forward_prefill_logits_all([5, 1, 4], 1)
    m.close()
    assert np.array_equal(got_one.view(np.uint32), np.resize(one, vocab).view(np.uint32))
    assert np.abs(got_many - np.stack([np.resize(r, vocab) for r in many])).max() <= 1e-5 * np.abs(many).max()   # splits of K may follow the row count


@pytest.mark.parametrize("vocab", ROWS)
@pytest.mark.parametrize("route", ["logit scale", "no decode copies"])
def test_one_row_by_the_copy(hip, base, route, vocab):
    """One position's logits where the head's launch does not write them into host memory itself."""
    cfg, weights, one, _ = base
    print(f"logits to host: {vocab} rows, {route}", flush=True)
    w = {**weights, **{name: _rows(weights[name], vocab) for name in ("token_embd.weight", "output.weight")}}
    scale = 4.0 if route == "logit scale" else 1.0
    m = hip_api.Model(hip, {**cfg, "vocab": vocab, "logit_scale": scale}, w)
    if route != "logit scale":
        m.drop_decode_copies()
    got = [m.forward(3, 0), m.forward_prefill([5, 1, 4], 1)]
    m.truncate_kv(0)
    again = [m.forward(3, 0), m.forward_prefill([5, 1, 4], 1)]
    m.close()
    assert np.array_equal(got[0].view(np.uint32), np.resize(one * np.float32(1 / scale), vocab).view(np.uint32))   # a power of two: exact
    assert all(np.array_equal(a.view(np.uint32), b.view(np.uint32)) for a, b in zip(got, again))
