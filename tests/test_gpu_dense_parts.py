"""256 x 256 tiles in parts of K where 128 x 128 ones would do with K whole: the reduction behind every epilogue that meets it, ragged
last parts, rows and tokens.  Whole small models against the reference; bars: those of the designs' own tests."""
import numpy as np
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


# gate | up, residual and head of a Nafevik; squared relu of a Fidinex
@pytest.mark.parametrize("family, width, ff, vocab, products", [("nafevik", 3072, 2016, 3001, [(4032, 3072), (3072, 2080), (3001, 3072)]), ("fidinex", 2060, 3072, 40, [(3072, 2060)])])
def test_no_room_for_the_parts(family, width, ff, vocab, products):
    """The sums of two parts do not fit into the context's workspace, and the smaller tiles take K whole: with room for less than one part's
    sums and for nearly two, the same bits, on contexts that have held no sums before."""
    n, out = 1290, []
    if family == "nafevik":
        cfg = N.config([N.attention(2, 1, 32, 32, 700, 32, 10000.0, ff=ff)], width=width, vocab=vocab, taps=2, positions=n)
        w = R.random_model(cfg, 79)
        toks, raw = N.tokens(cfg, n, 5), {k: v if k.endswith(TN.R_VECTORS) else N.bf16_bits(v) for k, v in w.items()}
        want, tol = N.reference(cfg, w, toks), TN.TOL[False]
    else:
        cfg = F.config([F.attention(2, 1, 32, 32, (0.3, 8), True, ff=ff)], width=width, vocab=vocab, streams=4)
        w = F.random_model(cfg, 83)
        toks, raw = F.tokens(cfg, n, 5), F.as_arrays(w)
        want, tol = F.reference(cfg, w, toks), TF.TOL[False]
    for limit in (12 << 20, 2 * min(rows for rows, _ in products) * n * 4 - 1):
        assert all(_in_parts(rows, k, n) and hip_api.dense_streams_tile(rows, k, n, 0, limit) == (128, 1) for rows, k in products)
        ctx = hip_api.Context(0)
        ctx.set_workspace_limit(limit)
        m = hip_api.LayeredModel(ctx, cfg, raw, n)
        print(f"no room for parts: {family}, limit {limit}", flush=True)
        out.append(m.forward_prefill_logits_all(toks, 0))
        m.close()
        ctx.close()
        print(f"no room for parts: {family}, limit {limit}: {N.rel(out[-1], want):.2e}", flush=True)
        assert N.rel(out[-1], want) < tol
    assert np.array_equal(out[0].view(np.uint32), out[1].view(np.uint32))
