"""The decode step's attention in one launch (short contexts) at the edges of its wavefronts' chunks of 16 keys and of its range, behind
which the two launches take over: against decode_attention on the rotated query and the completed cache, the appended rows and the
quantized outputs bit for bit.  Bar: sums of up to 321 f32 terms, 321 * 2^-24 = 2e-5 of the values' size."""
import numpy as np
import pytest

import util

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kv_f16", [False, True])
@pytest.mark.parametrize("n_heads,n_kv,hd", [(32, 8, 128), (24, 8, 128), (7, 1, 128), (3, 3, 64), (16, 2, 64)])
@pytest.mark.parametrize("keys", [1, 2, 15, 16, 17, 37, 113, 127, 128, 129, 145, 191, 192, 193, 257, 319, 320, 321])
def test_short_attention_step(hip, orc, kv_f16, n_heads, n_kv, hd, keys):
    print(f"short attention heads {n_heads}/{n_kv} of {hd}, {keys} keys, f16={kv_f16}", flush=True)
    pos, kv_dim = keys - 1, n_kv * hd
    q, k_new, v_new = util.make_x(n_heads * hd, 21 + pos), util.make_x(kv_dim, 22 + pos), util.make_x(kv_dim, 23 + pos)
    kc, vc = util.make_x(pos * kv_dim, 24), util.make_x(pos * kv_dim, 25)
    out, sc, qq, k_row, v_row = hip.attn_decode_step(q, k_new, v_new, kc, vc, n_heads, n_kv, hd, pos, 500000.0, norm=True, freq_factors=None, kv_f16=kv_f16)
    q_rot, k_rot = orc.rope(q, k_new, pos, n_heads, n_kv, hd, 500000.0, norm=True, freq_factors=None)

    def held(a):
        return a.astype(np.float16).astype(np.float32) if kv_f16 else a

    assert np.array_equal(k_row.view(np.uint32), held(k_rot).view(np.uint32)) and np.array_equal(v_row.view(np.uint32), held(v_new).view(np.uint32))
    ref = orc.decode_attention(q_rot, held(np.concatenate([kc, k_rot])), held(np.concatenate([vc, v_new])), n_heads, n_kv, hd, 1.0 / np.sqrt(hd), keys)
    assert np.abs(out - ref).max() <= 2e-5 * max(util.rms(ref), util.rms(v_new))
    rs, rq = orc.quantize_q8_0(out)
    assert np.array_equal(qq, rq) and np.array_equal(sc.view(np.uint32), rs.view(np.uint32))
