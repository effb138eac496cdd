"""The bf16 designs' decode products where a wavefront has one, two, three and more steps of weights, an input that is or is not whole in
the steps taken ahead, and attention's parts of more heads and columns than those: whole small models, token by token, against the
reference.  Bars: those of the designs' own tests."""
import pytest

import fidinex_util as U
from test_gpu_fidinex import DTYPES, TOL, _feed, _open

pytestmark = pytest.mark.gpu

# (width, ff, vocab, streams, heads, kv heads, head size)
SHAPES = [(96, 2100, 40, 4, 4, 2, 16),       # down: one step of a row
          (96, 5000, 40, 3, 4, 2, 16),       # two
          (100, 9000, 40, 4, 4, 2, 16),      # three
          (72, 13000, 40, 1, 4, 2, 16),      # four
          (64, 15300, 40, 4, 4, 2, 16),      # four, the longest input in 32 bits
          (70, 50, 40000, 4, 4, 2, 16),      # head: rows of one step, two and three groups of four a wavefront
          (1100, 64, 20000, 2, 4, 2, 16),    # two steps a row, one and two groups
          (2300, 64, 18000, 4, 4, 2, 16),    # three steps a row
          (4400, 600, 33, 4, 4, 2, 16),      # a norm of more columns than are taken ahead
          (160, 64, 40, 4, 40, 4, 8),        # parts of 40 heads
          (256, 64, 40, 4, 20, 2, 256)]      # 5120 columns of attention's result


@DTYPES
@pytest.mark.parametrize("width, ff, vocab, streams, heads, kv_heads, dim", SHAPES)
def test_steps_of_the_decode_products(tmp_path, width, ff, vocab, streams, heads, kv_heads, dim, f32):
    cfg = U.config([U.attention(heads, kv_heads, dim, dim, (0.3, 8), True, ff=ff)] * 2, width=width, vocab=vocab, streams=streams)
    w = U.random_model(cfg, 41)
    toks = U.tokens(cfg, 6, 3)
    m = _open(U.save(tmp_path / "m", cfg, w), f32)
    err = U.rel(_feed(m, toks, [1]), U.reference(cfg, w, toks))
    m.close()
    print(f"steps: width {width} ff {ff} vocab {vocab} heads {heads} of {dim} f32={f32}: {err:.2e}", flush=True)
    assert err < TOL[f32]
