"""Sums of the residual streams with the next norm behind them: rows of one to several groups of four channels a thread, a width that is
no multiple of four, one whose row the workgroup's LDS does not hold, no more tokens than compute units and more.  Bars: those of the
design's own tests."""
import pytest

import fidinex_util as U
from test_gpu_fidinex import DTYPES, TOL, _feed, _open

pytestmark = pytest.mark.gpu

# (width, streams, tokens)
SHAPES = [(50, 3, 40), (254, 4, 70), (2050, 3, 33), (2052, 2, 300), (4100, 8, 20), (4098, 4, 257), (16384, 3, 17), (16400, 3, 17)]


@DTYPES
@pytest.mark.parametrize("width, streams, n", SHAPES)
def test_streams_with_the_next_norm(tmp_path, width, streams, n, f32):
    cfg = U.config([U.attention(4, 2, 16, 16, (0.3, 8), True, ff=72), U.latent(2, 16, 8, 16, 24, 100.0), U.attention(4, 2, 16, 16, None, True, ff=40)],
                   width=width, vocab=37, streams=streams)
    w = U.random_model(cfg, 53)
    toks = U.tokens(cfg, n, 7)
    m = _open(U.save(tmp_path / "m", cfg, w), f32)
    err = U.rel(_feed(m, toks, [n]), U.reference(cfg, w, toks))
    m.close()
    print(f"streams and norm: width {width}, {streams} streams, {n} tokens f32={f32}: {err:.2e}", flush=True)
    assert err < TOL[f32]
