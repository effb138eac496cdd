"""256 x 256 tiles in parts of K where 128 x 128 ones would do with K whole: the reduction behind every epilogue that meets it, ragged
last parts, rows and tokens.  Whole small models against the reference; bars: those of the designs' own tests."""
import pytest

import fidinex_util as F
import nafevik_ref as R
import nafevik_util as N
import test_gpu_fidinex as TF
import test_gpu_nafevik as TN
from cera_amd import hip_api

pytestmark = pytest.mark.gpu


def _in_parts(rows, k, n, streams=0):
    tile, parts = hip_api.dense_streams_tile(rows, k, n, streams)
    return hip_api.dense_tile(rows, k, n) == 128 and tile == 256 and parts > 1


# residual products in eight and five parts; gate | up and the head of all positions in two, residual in one
@pytest.mark.parametrize("width, ff, n, vocab, products", [(1500, 8200, 700, 64, [(1500, 8264)]), (1100, 9001, 1501, 50, [(1100, 9065)]),
                                                           (2060, 1504, 1290, 3001, [(3008, 2060), (3001, 2060)])])
def test_residual_swiglu_and_plain_sums(tmp_path, width, ff, n, vocab, products):
    assert all(_in_parts(rows, k, n) for rows, k in products)
    cfg = N.config([N.attention(2, 1, 32, 32, 700, 32, 10000.0, ff=ff)], width=width, vocab=vocab, taps=2, positions=n)
    w = R.random_model(cfg, 71)
    m = TN._open(N.save(tmp_path / "m", cfg, w), False, n)
    toks = N.tokens(cfg, n, 5)
    err = N.rel(m.forward_prefill_logits_all(toks, 0), N.reference(cfg, w, toks))
    m.close()
    print(f"parts: width={width} ff={ff} n={n}: {err:.2e}", flush=True)
    assert err < TN.TOL[False]


@pytest.mark.parametrize("width, ff, n, streams, product", [(2060, 3001, 1290, 4, (3001, 2060, 1290, 0)), (1500, 8200, 700, 3, (1500, 8200, 700, 3)), (1500, 8200, 700, 4, (1500, 8200, 700, 4))])
def test_squared_relu_and_streams(tmp_path, width, ff, n, streams, product):
    assert _in_parts(*product)
    cfg = F.config([F.attention(2, 1, 32, 32, (0.3, 8), True, ff=ff)], width=width, vocab=40, streams=streams)
    w = F.random_model(cfg, 73)
    m = TF._open(F.save(tmp_path / "m", cfg, w), False, n)
    toks = F.tokens(cfg, n, 7)
    err = F.rel(m.forward_prefill_logits_all(toks, 0), F.reference(cfg, w, toks))
    m.close()
    print(f"parts: width={width} ff={ff} streams={streams}: {err:.2e}", flush=True)
    assert err < TF.TOL[False]
