"""The first step behind a prompt or a cut, whose launch of the embedding adds up every layer's convolution history: rows of one and of
several workgroups, few and many taps, fewer positions than taps, layers with one convolution and with two, passes of a loop."""
import numpy as np
import pytest

import nafevik_ref as R
import nafevik_util as U
from test_gpu_nafevik import DTYPES, TOL, _feed, _open

pytestmark = pytest.mark.gpu


@DTYPES
@pytest.mark.parametrize("width, taps, loop", [(48, 2, None), (300, 9, (1, 3, 2)), (520, 4, None)])
def test_first_steps(tmp_path, width, taps, loop, f32):
    layers = [U.attention(2, 2, 16, 16, 30, 16, 100.0, ff=32), U.attention(4, 2, 16, 24, None, 16, 100.0), U.attention(2, 1, 16, 16, 40, 8, 100.0, ff=72)]
    cfg = U.config(layers, width=width, vocab=30, taps=taps, **({"loop": loop} if loop else {}))
    w = R.random_model(cfg, 83)
    m = _open(U.save(tmp_path / "m", cfg, w), f32)
    toks = np.random.default_rng(5).integers(0, 30, 90)
    want = U.reference(cfg, w, toks)
    for cuts in ([2, 1, 1], [7, 1], [60, 1, 2, 1]):
        assert U.rel(_feed(m, toks, cuts), want) < TOL[f32], cuts
    m.truncate_kv(80)
    got = [m.forward(int(toks[p]), p) for p in (80, 81)]
    assert U.rel(np.stack(got), want[80:82]) < TOL[f32]
    m.close()
