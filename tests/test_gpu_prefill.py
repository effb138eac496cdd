"""GPU parity for the prefill path: int8-MFMA GEMM vs the oracle's gemm_preq on
the same Q8_0-quantized activations, and batched prefill of a small llama vs
the oracle's forward_prefill_batched."""
import numpy as np
import pytest

import util
from util import Q4_0, Q4_1, Q8_0, Q4_K, Q5_K, Q6_K
from cera_amd import hip_api, synth

pytestmark = pytest.mark.gpu
GEMM_TOL = 1e-3  # x rms(ref), the north star's bar for GEMM


def _say(msg):
    print(msg, flush=True)


def _oracle_gemm(orc, dtype, w, x, m, n, k):
    bs = np.empty((n, k // 32), np.float32)
    bq = np.empty((n, k), np.int8)
    for j in range(n):
        bs[j], bq[j] = orc.quantize_q8_0(x[j])
    return orc.gemm_preq(dtype, w, bs, bq, m, n, k)


@pytest.mark.parametrize("dtype", util.INT8_TYPES)
@pytest.mark.parametrize("m,n,k", [(128, 64, 256), (7, 3, 512), (200, 65, 1024), (130, 1, 256), (64, 130, 4096)])
def test_gemm_small_shapes(hip, orc, dtype, m, n, k):
    _say(f"gemm {util.NAMES[dtype]} m={m} n={n} k={k}")
    w, _ = util.make_weights(dtype, m, k, seed=dtype * 10 + m)
    x = util.rng(dtype + n).standard_normal((n, k)).astype(np.float32)
    out = hip.gemm(dtype, w, x, m, n, k)
    ref = _oracle_gemm(orc, dtype, w, x, m, n, k)
    err = np.abs(out.astype(np.float64) - ref).max()
    assert err <= GEMM_TOL * util.rms(ref), (err, util.rms(ref))


@pytest.mark.parametrize("dtype", util.INT8_TYPES)
def test_gemm_seeded_shape_sweep(hip, orc, dtype):
    """Seeded random (rows, tokens, k): ragged tiles on both sides, and few output tiles with a long
    K so the split-K route and its fixed-order reduction are exercised."""
    r = util.rng(5000 + dtype)
    shapes = [(int(r.integers(1, 400)), int(r.integers(1, 200)), 256 * int(r.integers(1, 17))) for _ in range(5)]
    shapes += [(64, 48, 8192), (130, 17, 14336), (256, 64, 4096)]
    for m, n, k in shapes:
        _say(f"gemm sweep {util.NAMES[dtype]} m={m} n={n} k={k}")
        w, _ = util.make_weights(dtype, m, k, seed=dtype * 7 + m)
        x = util.rng(m + n).standard_normal((n, k)).astype(np.float32)
        out = hip.gemm(dtype, w, x, m, n, k)
        ref = _oracle_gemm(orc, dtype, w, x, m, n, k)
        err = np.abs(out.astype(np.float64) - ref).max()
        assert err <= GEMM_TOL * util.rms(ref), (m, n, k, err, util.rms(ref))


@pytest.mark.parametrize("dtype,m,k", [(Q4_K, 4096, 4096), (Q6_K, 4096, 14336)])
@pytest.mark.parametrize("n", [128, 512, 2048])
def test_gemm_config3_shapes_row_sample(hip, orc, dtype, m, k, n):
    """BASELINE config 3 shapes; the oracle checks a sample of output rows."""
    _say(f"gemm {util.NAMES[dtype]} m={m} n={n} k={k}")
    w, _ = util.make_weights(dtype, m, k, seed=3)
    x = util.rng(n).standard_normal((n, k)).astype(np.float32)
    out = hip.gemm(dtype, w, x, m, n, k)
    rows = np.unique(np.concatenate([np.arange(8), util.rng(1).integers(0, m, 40), np.arange(m - 8, m)]))
    rb = util.H.row_bytes(dtype, k)
    wr = np.ascontiguousarray(w.reshape(m, rb)[rows]).reshape(-1)
    ref = _oracle_gemm(orc, dtype, wr, x, rows.size, n, k)
    err = np.abs(out[rows].astype(np.float64) - ref).max()
    assert err <= GEMM_TOL * util.rms(ref), (err, util.rms(ref))


def test_gemm_equals_gemv_per_column(hip, orc):
    """decode == prefill at the GEMM level: every column of the GEMM agrees with the
    GEMV of that token (tests/avx2_decode_prefill_identity.rs, to the float bar)."""
    m, n, k = 96, 5, 1024
    for dtype in (Q4_K, Q6_K, Q4_0):
        w, _ = util.make_weights(dtype, m, k, seed=9)
        x = util.rng(7).standard_normal((n, k)).astype(np.float32)
        out = hip.gemm(dtype, w, x, m, n, k)
        for j in range(n):
            y = hip.gemv(dtype, w, x[j], m, k)
            assert np.abs(out[:, j] - y).max() <= 2e-5 * max(util.rms(y), 1e-6) * 10


@pytest.mark.parametrize("dtype", [Q4_K, Q6_K, Q4_0])
@pytest.mark.parametrize("ma,mb,n,k", [(256, 128, 40, 512), (4096, 1024, 512, 4096), (300, 77, 33, 2048),
                                       (1024, 1024, 1100, 256)])
def test_gemm_pair_matches_single_launches(hip, orc, dtype, ma, mb, n, k):
    """Q|K and gate|up share a launch in the prefill pass: each output equals the matrix's own GEMM
    (bit for bit where neither launch splits K; to the order of the partial sums where they do,
    as at 4096 x 4096 | 1024 x 4096 with 512 tokens), and a row sample agrees with the oracle."""
    _say(f"gemm pair {util.NAMES[dtype]} ma={ma} mb={mb} n={n} k={k}")
    wa, _ = util.make_weights(dtype, ma, k, seed=31)
    wb, _ = util.make_weights(dtype, mb, k, seed=32)
    x = util.rng(n + k).standard_normal((n, k)).astype(np.float32)
    oa, ob = hip.gemm_pair(dtype, wa, ma, dtype, wb, mb, x, n, k)
    sa, sb = hip.gemm(dtype, wa, x, ma, n, k).T, hip.gemm(dtype, wb, x, mb, n, k).T
    for got, single in ((oa, sa), (ob, sb)):
        assert np.abs(got - single).max() <= 2e-5 * util.rms(single)
    rows = np.unique(np.concatenate([np.arange(4), np.arange(mb - 4, mb)]))
    rb = util.H.row_bytes(dtype, k)
    wr = np.ascontiguousarray(wb.reshape(mb, rb)[rows]).reshape(-1)
    ref = _oracle_gemm(orc, dtype, wr, x, rows.size, n, k)
    assert np.abs(ob[:, rows].T.astype(np.float64) - ref).max() <= GEMM_TOL * util.rms(ref)


@pytest.mark.parametrize("dtype", [Q4_K, Q6_K])
@pytest.mark.parametrize("ma,mb,k", [(300, 68, 2048), (64, 4, 2304), (132, 1024, 14336)])
@pytest.mark.parametrize("n", [2, 5, 16, 17, 32, 33, 48])
def test_gemm_pair_of_a_few_tokens(hip, orc, dtype, ma, mb, k, n):
    """Two to 48 tokens against the exact product of the dequantized weights and quantized tokens: block results are whole
    numbers, so what is left is the rounding of k / 32 sums, sqrt(448) 2^-24 of a partial sum or about 1.3e-6 of the outputs'
    rms at the longest row, and 2e-5 is fifteen times that.  Last tiles of rows and tokens, one to four tokens of a last tile,
    slices of K that do not divide into the chunks read ahead; the native
    bytes give the same bits as the decode copy."""
    _say(f"few tokens {util.NAMES[dtype]} ma={ma} mb={mb} k={k} n={n}")
    wa, _ = util.make_weights(dtype, ma, k, seed=51)
    wb, _ = util.make_weights(dtype, mb, k, seed=52)
    x = util.rng(n + k).standard_normal((n, k)).astype(np.float32) * np.exp2(util.rng(n).integers(-6, 7, (n, 1))).astype(np.float32)
    xs, xq = orc.quantize_q8_0(x.reshape(-1))
    xd = (xq.reshape(-1, 32).astype(np.float64) * xs.reshape(-1, 1)).reshape(n, k)
    oa, ob = hip.gemm_pair(dtype, wa, ma, dtype, wb, mb, x, n, k)
    hip.set_decode_copies(False)
    try:
        native = hip.gemm_pair(dtype, wa, ma, dtype, wb, mb, x, n, k)
    finally:
        hip.set_decode_copies(True)
    assert np.array_equal(oa, native[0]) and np.array_equal(ob, native[1])
    for got, w, m in ((oa, wa, ma), (ob, wb, mb)):
        want = xd @ util.dequant_np(dtype, w, m, k).astype(np.float64).T
        rms = np.sqrt(np.mean(want * want, axis=1, keepdims=True))
        assert (np.abs(got - want) / rms).max() <= 2e-5


@pytest.mark.parametrize("ma,mb,n,k", [(200, 56, 66, 14336), (1, 4, 68, 14336), (256, 256, 128, 4352), (260, 17, 132, 14336),
                                       (1028, 4, 257, 2304), (1028, 300, 256, 4096), (2052, 256, 2049, 1024)])
def test_gemm_q6k_of_many_tokens(hip, orc, ma, mb, n, k):
    """Q6_K with more than 64 tokens against the exact product of the dequantized weights and quantized tokens, alone (one
    output row after the other) and as a pair (one token after the other): last tiles of rows and tokens, one row, one to
    sixteen slices of K from one super-block on.  Scales and codes of random bytes take the whole range, -128 times -32
    included, so both parts of a weight count; the bound is that of the products of a few tokens above, of an output's rms
    over random signs."""
    _say(f"many tokens Q6_K ma={ma} mb={mb} n={n} k={k}")
    r = util.rng(ma + n + k)
    def weights(m):
        w = r.integers(0, 256, (m, k // 256, 210), dtype=np.uint8)
        w[:, :, 208:] = (r.uniform(0.5, 2.0, (m, k // 256, 1)) * 1e-3).astype(np.float16).view(np.uint8)
        return w.reshape(-1)
    wa, wb = weights(ma), weights(mb)
    x = r.standard_normal((n, k)).astype(np.float32) * np.exp2(r.integers(-6, 7, (n, 1))).astype(np.float32)
    xs, xq = orc.quantize_q8_0(x.reshape(-1))
    xd = (xq.reshape(-1, 32).astype(np.float64) * xs.reshape(-1, 1)).reshape(n, k)
    alone = hip.gemm(Q6_K, wa, x, ma, n, k)
    oa, ob = hip.gemm_pair(Q6_K, wa, ma, Q6_K, wb, mb, x, n, k)
    for got, w, m in ((alone.reshape(ma, n).T, wa, ma), (oa, wa, ma), (ob, wb, mb)):
        wd = util.dequant_np(Q6_K, w, m, k).astype(np.float64)
        rms = np.sqrt((xd * xd).sum(1, keepdims=True) * (wd * wd).sum(1) / k)
        assert (np.abs(got - xd @ wd.T) / rms).max() <= 2e-5


@pytest.mark.parametrize("dtype,bytes_", [(Q8_0, 34), (Q4_0, 18)])
@pytest.mark.parametrize("ma,mb,n,k", [(1, 4, 65, 256), (127, 129, 68, 512), (128, 36, 128, 8192), (260, 17, 132, 2304),
                                       (1028, 300, 257, 4096), (132, 2052, 1001, 1024), (5, 64, 4, 256), (130, 62, 64, 2304), (36, 4, 33, 8192)])
def test_gemm_of_32_weight_blocks(hip, orc, dtype, bytes_, ma, mb, n, k):
    """Q8_0 and Q4_0 against the exact product of the dequantized weights and quantized tokens, alone and as a pair: tiles of
    64 and of 128 tokens, last tiles of rows and tokens, one row, one to eight slices of K.  Codes are random bytes, -128 and -8
    among them, scales have both signs; the bound is that of the products of a few tokens above, of an output's rms over
    random signs."""
    _say(f"many tokens {util.NAMES[dtype]} ma={ma} mb={mb} n={n} k={k}")
    r = util.rng(ma + n + k)
    def weights(m):
        w = r.integers(0, 256, (m, k // 32, bytes_), dtype=np.uint8)
        d = r.uniform(0.5, 2.0, (m, k // 32, 1)) * 1e-3 * r.choice([-1.0, 1.0], (m, k // 32, 1))
        w[:, :, :2] = d.astype(np.float16).view(np.uint8)
        return w.reshape(-1)
    wa, wb = weights(ma), weights(mb)
    x = r.standard_normal((n, k)).astype(np.float32) * np.exp2(r.integers(-6, 7, (n, 1))).astype(np.float32)
    xs, xq = orc.quantize_q8_0(x.reshape(-1))
    xd = (xq.reshape(-1, 32).astype(np.float64) * xs.reshape(-1, 1)).reshape(n, k)
    alone = hip.gemm(dtype, wa, x, ma, n, k)
    oa, ob = hip.gemm_pair(dtype, wa, ma, dtype, wb, mb, x, n, k)
    for got, w, m in ((alone.reshape(ma, n).T, wa, ma), (oa, wa, ma), (ob, wb, mb)):
        wd = util.dequant_np(dtype, w, m, k).astype(np.float64)
        rms = np.sqrt((xd * xd).sum(1, keepdims=True) * (wd * wd).sum(1) / k)
        assert (np.abs(got - xd @ wd.T) / rms).max() <= 2e-5


@pytest.mark.parametrize("dtype,bytes_", [(Q8_0, 34), (Q4_0, 18)])
@pytest.mark.parametrize("n", [40, 130])
def test_gemm_of_32_weight_blocks_with_subnormal_scales(hip, orc, dtype, bytes_, n):
    """Weights' and tokens' scales below 2^-14, subnormal as f16, in the outer product on the matrix core: it keeps them, and a
    product of two is exact in f32.  One row's scales are the smallest there are; bound as above."""
    m, k = 132, 1024
    _say(f"subnormal scales {util.NAMES[dtype]} n={n}")
    r = util.rng(n)
    w = r.integers(0, 256, (m, k // 32, bytes_), dtype=np.uint8)
    d = (r.uniform(0.5, 2.0, (m, k // 32, 1)) * 1e-5).astype(np.float16)
    d[0] = np.float16(2.0 ** -24)
    w[:, :, :2] = d.view(np.uint8)
    x = (r.standard_normal((n, k)) * 2.0 ** -10).astype(np.float32)
    xs, xq = orc.quantize_q8_0(x.reshape(-1))
    assert 0 < xs.min() and xs.max() < 2.0 ** -14
    xd = (xq.reshape(-1, 32).astype(np.float64) * xs.reshape(-1, 1)).reshape(n, k)
    wd = util.dequant_np(dtype, w.reshape(-1), m, k).astype(np.float64)
    rms = np.sqrt((xd * xd).sum(1, keepdims=True) * (wd * wd).sum(1) / k)
    got = hip.gemm(dtype, w.reshape(-1), x, m, n, k).reshape(m, n).T
    assert (np.abs(got - xd @ wd.T) / rms).max() <= 2e-5


@pytest.mark.parametrize("dtype,bytes_", [(Q8_0, 34), (Q4_0, 18)])
def test_gemm_of_rows_of_16_million_columns(hip, orc, dtype, bytes_):
    """Rows that the kernel of the other Q8_0 and Q4_0 products has no offsets for.  A slice of K adds 2^16 blocks one after the other:
    roundings of at most 2^-24 of sums that grow as a random walk come to 2^-24 * sqrt(2^16 / 6) of the output's rms; 2.5 times that."""
    m, n, k = 4, 2, 1 << 24
    _say(f"{util.NAMES[dtype]} m={m} k={k} n={n}")
    r = util.rng(bytes_)
    w = r.integers(0, 256, (m, k // 32, bytes_), dtype=np.uint8)
    d = r.uniform(0.5, 2.0, (m, k // 32, 1)).astype(np.float32) * r.choice(np.float32([-1e-3, 1e-3]), (m, k // 32, 1))
    w[:, :, :2] = d.astype(np.float16).view(np.uint8)
    x = r.standard_normal((n, k), dtype=np.float32)
    xs, xq = orc.quantize_q8_0(x.reshape(-1))
    xd = (xq.reshape(-1, 32).astype(np.float64) * xs.reshape(-1, 1)).reshape(n, k)
    wd = util.dequant_np(dtype, w.reshape(-1), m, k).astype(np.float64)
    rms = np.sqrt((wd * wd).sum(1, keepdims=True) * (xd * xd).sum(1) / k)
    assert (np.abs(hip.gemm(dtype, w.reshape(-1), x, m, n, k) - wd @ xd.T) / rms).max() <= 2.0 ** -16


@pytest.mark.parametrize("dtype,m,k,n", [(Q4_K, 132, 2304, 5), (Q4_K, 300, 4096, 48), (Q6_K, 132, 2304, 3), (Q6_K, 300, 4096, 33),
                                         (Q6_K, 300, 4096, 160), (Q6_K, 516, 2304, 384), (Q8_0, 132, 2304, 9), (Q8_0, 300, 4096, 64), (Q8_0, 516, 2304, 200),
                                         (Q4_0, 132, 2304, 9), (Q4_0, 300, 4096, 64), (Q4_0, 516, 2304, 200)])
def test_block_results_are_whole_numbers(hip, dtype, m, k, n):
    """The products of a few and of many tokens in the kernels that passes run: tokens of a single block each and scales
    that are powers of two leave one block's whole number in every output, so any rounding on the way would show.  Weights
    of random bytes take the whole range; the last row's scales and codes and the first token's quants are the largest, 32
    of -128 * -32 * 127 for Q6_K, 1 % below 2^24, and of -128 * 127 for Q8_0, whose sums leave the matrix cores as floats."""
    _say(f"whole numbers {util.NAMES[dtype]} m={m} k={k} n={n}")
    r = util.rng(m + n)
    bytes_ = {Q4_K: 144, Q6_K: 210, Q8_0: 8 * 34, Q4_0: 8 * 18}[dtype]
    w = r.integers(0, 256, (m, k // 256, bytes_), dtype=np.uint8)
    w[-1] = {Q4_K: 255, Q6_K: 0, Q8_0: 128, Q4_0: 0}[dtype]     # the largest scales, mins and codes; for Q6_K code 0 is -32, for Q4_0 -8
    if dtype == Q6_K:
        w[-1, :, 192:208] = 128
    d = np.exp2(r.integers(-12, -5, (m, k // 256, 1))).astype(np.float16).view(np.uint8)
    if dtype == Q4_K:
        w[:, :, 0:2], w[:, :, 2:4] = d, d
    elif dtype == Q6_K:
        w[:, :, 208:210] = d
    else:
        w.reshape(m, k // 32, -1)[:, :, :2] = np.exp2(r.integers(-12, -5, (m, k // 32, 1))).astype(np.float16).view(np.uint8)
    x = np.zeros((n, k // 32, 32), np.float32)
    for t in range(n):
        q = r.integers(-127, 128, 32) if t else np.full(32, 127)
        q[t % 32] = 127                     # so that the block's scale is a power of two
        x[t, t * 7 % (k // 32)] = q * np.exp2(int(r.integers(-8, 9)))
    x = x.reshape(n, k)
    want = (x.astype(np.float64) @ util.dequant_np(dtype, w.reshape(-1), m, k).astype(np.float64).T).astype(np.float32)
    for copies in (True, False):
        hip.set_decode_copies(copies)
        try:
            got = hip.gemm_pair(dtype, w.reshape(-1), m, dtype, w.reshape(-1), m, x, n, k)
        finally:
            hip.set_decode_copies(True)
        assert np.array_equal(got[0], want) and np.array_equal(got[1], want), copies
    if n > 64:
        assert np.array_equal(hip.gemm(dtype, w.reshape(-1), x, m, n, k).reshape(m, n).T, want)


@pytest.mark.parametrize("dtype,n,m,k,limit", [(Q4_K, 48, 4096, 2048, 2 << 20), (Q6_K, 5, 4096, 2048, 1 << 18), (Q6_K, 128, 4096, 2048, 4 << 20)])
def test_products_without_room_for_partial_sums(dtype, n, m, k, limit):
    """Sums over parts of K are a workspace that a product can do without: where it cannot be had (here by a limit that the
    inputs and outputs fit and the parts do not), one workgroup takes the whole of K.  Both are within 2e-5 of the outputs' rms
    of the exact product, as test_gemm_pair_of_a_few_tokens has it."""
    w, _ = util.make_weights(dtype, m, k, seed=3)
    x = util.rng(n).standard_normal((n, k)).astype(np.float32)
    out = []
    for room in (0, limit):
        ctx = hip_api.Context(0)
        ctx.set_workspace_limit(room)
        _say(f"gemm_pair {util.NAMES[dtype]} {m}x{k} n={n} limit {room}")
        out.append(ctx.gemm_pair(dtype, w, m, dtype, w, m, x, n, k))
        ctx.close()
    assert np.array_equal(out[1][0], out[1][1])
    assert np.abs(out[0][0] - out[1][0]).max() <= 4e-5 * util.rms(out[0][0])


@pytest.mark.parametrize("dtype", [Q4_K, Q4_0, Q4_1, Q8_0])
@pytest.mark.parametrize("m,k,n,want_fused", [(2048, 512, 1040, True), (1056, 256, 2000, True), (512, 256, 70, False), (32800, 256, 33, True)])
def test_gemm_swiglu_epilogue_matches_separate_kernels(hip, orc, dtype, m, k, n, want_fused):
    """gate | up | SwiGLU | Q8_0 in one launch: the quants and scales must be, byte for byte, the
    oracle's quantization of the oracle's SwiGLU of the two GEMM outputs the pair launch gives
    (silu_mul_inplace cpu.rs:2570-2575, quantize_columns transformer.rs:865-946).  Row counts
    that are not a multiple of the 64-row tile, ragged token tiles, and a batch too small to
    fill the chip (which takes the separate kernels) are covered."""
    _say(f"gemm_swiglu {util.NAMES[dtype]} m={m} k={k} n={n}")
    wg, _ = util.make_weights(dtype, m, k, seed=41)
    wu, _ = util.make_weights(dtype, m, k, seed=42)
    x = util.rng(m + 3 * n).standard_normal((n, k)).astype(np.float32)
    q, sc, fused = hip.gemm_swiglu(dtype, wg, wu, m, x, n, k)
    assert fused == want_fused
    g, u = hip.gemm_pair(dtype, wg, m, dtype, wu, m, x, n, k)
    h = orc.silu_mul(g.reshape(-1), u.reshape(-1))
    ref_s, ref_q = orc.quantize_q8_0(h)
    assert np.array_equal(q.reshape(-1), ref_q)
    assert np.array_equal(sc.reshape(-1).view(np.uint32), ref_s.view(np.uint32))


@pytest.mark.parametrize("m,n,k", [(12801, 449, 512), (12800, 512, 256), (12928, 511, 768)])
def test_gemm_q4k_by_128_tokens(hip, orc, m, n, k):
    """Q4_K launches that take workgroups of 128 tokens (two rounds of the chip by 64, one by 128): a last tile of 128 tokens with
    nothing in its upper half, a whole one, a ragged one; whole and ragged tiles of rows.  A token's bits are those of a launch of
    64 tokens, which takes 64 a workgroup (K is whole in both); the pair of halves and its SwiGLU launch agree byte for byte."""
    _say(f"gemm Q4_K by 128 tokens m={m} n={n} k={k}")
    w, _ = util.make_weights(Q4_K, m, k, seed=61)
    x = util.rng(n + k).standard_normal((n, k)).astype(np.float32)
    out = hip.gemm(Q4_K, w, x, m, n, k)
    for a in (0, 64, (n - 1) // 64 * 64):
        part = x[a:a + 64]
        assert np.array_equal(out[:, a:a + 64].view(np.uint32), hip.gemm(Q4_K, w, part, m, len(part), k).view(np.uint32))
    h, rb = m // 64 * 32, util.H.row_bytes(Q4_K, k)
    wg, wu = w[:h * rb], w[h * rb:2 * h * rb]
    g, u = hip.gemm_pair(Q4_K, wg, h, Q4_K, wu, h, x, n, k)
    assert np.array_equal(g.T, out[:h]) and np.array_equal(u.T, out[h:2 * h])
    q, sc, fused = hip.gemm_swiglu(Q4_K, wg, wu, h, x, n, k)
    ref_s, ref_q = orc.quantize_q8_0(orc.silu_mul(g.reshape(-1), u.reshape(-1)))
    assert fused and np.array_equal(q.reshape(-1), ref_q) and np.array_equal(sc.reshape(-1).view(np.uint32), ref_s.view(np.uint32))


@pytest.mark.parametrize("n", [897, 900, 960])
def test_gemm_q4k_by_128_tokens_in_parts_of_k(hip, orc, n):
    """4096 x 4096 with 15 tiles of 64 tokens: two slices of K, two rounds of the chip by 64 tokens and one by 128.  Against the exact products
    of the dequantized weights and quantized tokens; block results are whole numbers, and the bound is that of test_gemm_pair_of_a_few_tokens."""
    m = k = 4096
    _say(f"gemm Q4_K by 128 tokens in parts n={n}")
    w, _ = util.make_weights(Q4_K, m, k, seed=62)
    x = util.rng(n).standard_normal((n, k)).astype(np.float32)
    xs, xq = orc.quantize_q8_0(x.reshape(-1))
    xd = (xq.reshape(-1, 32).astype(np.float64) * xs.reshape(-1, 1)).reshape(n, k)
    want = xd @ util.dequant_np(Q4_K, w, m, k).astype(np.float64).T
    rms = np.sqrt(np.mean(want * want, axis=1, keepdims=True))
    assert (np.abs(hip.gemm(Q4_K, w, x, m, n, k).T - want) / rms).max() <= 2e-5


@pytest.mark.parametrize("dtype", [Q4_K, Q6_K])
@pytest.mark.parametrize("m,k,n,want_fused", [(12288, 2048, 2, True), (12320, 2304, 5, True), (12288, 2048, 16, True), (12320, 2048, 17, True), (12288, 2048, 48, True), (96, 2048, 5, True), (4096, 2048, 48, False)])
def test_gemm_swiglu_of_a_few_tokens(hip, orc, dtype, m, k, n, want_fused):
    """As test_gemm_swiglu_epilogue_matches_separate_kernels for the kernel of 2 to 48 tokens: a last workgroup of 32 rows, one to
    three tiles of tokens, whole and not; the quants and scales are the oracle's of the two products of the pair launch."""
    _say(f"few gemm_swiglu {util.NAMES[dtype]} m={m} k={k} n={n}")
    wg, _ = util.make_weights(dtype, m, k, seed=41)
    wu, _ = util.make_weights(dtype, m, k, seed=42)
    x = util.rng(m + 3 * n).standard_normal((n, k)).astype(np.float32)
    q, sc, fused = hip.gemm_swiglu(dtype, wg, wu, m, x, n, k)
    assert fused == want_fused
    if not fused:
        return
    g, u = hip.gemm_pair(dtype, wg, m, dtype, wu, m, x, n, k)
    ref_s, ref_q = orc.quantize_q8_0(orc.silu_mul(g.reshape(-1), u.reshape(-1)))
    assert np.array_equal(q.reshape(-1), ref_q) and np.array_equal(sc.reshape(-1).view(np.uint32), ref_s.view(np.uint32))


@pytest.mark.parametrize("dtype", [Q4_K, Q6_K])
@pytest.mark.parametrize("n", [3, 5, 12, 16, 20, 45])
def test_gemm_swiglu_of_a_few_tokens_with_long_rows(hip, orc, dtype, n):
    """The whole of a long K in one workgroup, many chunks of tokens one after the other in the same two buffers, against the exact products
    of the dequantized weights and quantized tokens.  A product is off by at most 2e-5 of its token's rms (test_gemm_pair_of_a_few_tokens),
    |d silu / dg| <= 1.1 and |silu(g)| <= |g|; a quant is off by half a step d, d's f16 by 2^-11 of up to 127 steps."""
    m, k, distinct = 12288, 14336, 96
    _say(f"few gemm_swiglu, long rows {util.NAMES[dtype]} n={n}")
    (wg, _), (wu, _) = (util.make_weights(dtype, distinct, k, seed=s) for s in (43, 44))
    x = util.rng(n).standard_normal((n, k)).astype(np.float32)
    xs, xq = orc.quantize_q8_0(x.reshape(-1))
    xd = (xq.reshape(-1, 32).astype(np.float64) * xs.reshape(-1, 1)).reshape(n, k)
    g, u = (xd @ util.dequant_np(dtype, w, distinct, k).astype(np.float64).T for w in (wg, wu))
    h = g / (1 + np.exp(-g)) * u
    off = 2e-5 * (1.1 * np.abs(u) * util.rms(g) + np.abs(g) * util.rms(u)) + 1e-6 * np.abs(h)
    q, sc, fused = hip.gemm_swiglu(dtype, np.tile(wg, m // distinct), np.tile(wu, m // distinct), m, x, n, k)
    assert fused
    d = sc.reshape(n, m // distinct, distinct // 32, 1).astype(np.float64)
    got = (q.reshape(n, m // distinct, distinct // 32, 32) * d).reshape(n, m // distinct, distinct)
    assert (np.abs(got - h[:, None]) <= off[:, None] + (0.5 + 127 / 2048) * np.repeat(d, 32, 3).reshape(got.shape)).all()


@pytest.mark.parametrize("dtype,m,k,n,want_fused", [(Q4_K, 2048, 512, 1040, True), (Q4_K, 1056, 256, 2000, True),
                                                      (Q4_K, 6400, 256, 449, True), (Q4_K, 6400, 256, 510, True),   # by 128 tokens
                                                      (Q4_K, 512, 256, 80, False), (Q4_0, 2048, 512, 1040, True)])
def test_gemm_swiglu_f16_words_for_a_q6k_down_projection(hip, dtype, m, k, n, want_fused):
    """The f16 form of the SwiGLU quants that a Q6_K down projection reads: half words of the integer
    quants, every four in the order 0, 2, 1, 3 -- whether the Q4_K epilogue writes them or the
    conversion kernel makes them from the quants afterwards (small batches, other types)."""
    _say(f"gemm_swiglu_f16 {util.NAMES[dtype]} m={m} k={k} n={n}")
    wg, _ = util.make_weights(dtype, m, k, seed=43)
    wu, _ = util.make_weights(dtype, m, k, seed=44)
    x = util.rng(m + 5 * n).standard_normal((n, k)).astype(np.float32)
    q, sc, hv, fused = hip.gemm_swiglu_f16(dtype, wg, wu, m, x, n, k)
    assert fused == want_fused
    q0, sc0, _ = hip.gemm_swiglu(dtype, wg, wu, m, x, n, k)
    assert np.array_equal(q, q0) and np.array_equal(sc.view(np.uint32), sc0.view(np.uint32))
    want = q.astype(np.float16).reshape(-1, 4)[:, [0, 2, 1, 3]].reshape(n, m)
    assert np.array_equal(hv, want.view(np.uint16))


def test_gemm_pair_refuses_mixed_types(hip):
    with pytest.raises(hip_api.HipError) as e:
        hip.gemm_pair(Q4_K, np.zeros(144 * 4, np.uint8), 4, Q6_K, np.zeros(210 * 4, np.uint8), 4,
                      np.zeros((4, 256), np.float32), 4, 256)
    assert e.value.status == 3


def test_gemm_refuses_unsupported(hip):
    with pytest.raises(hip_api.HipError) as e:  # Q5_K has no Q8_0 route: no paired / SwiGLU / block-dot entry
        hip.gemm_pair(Q5_K, np.zeros(176 * 4, np.uint8), 4, Q5_K, np.zeros(176 * 4, np.uint8), 4,
                      np.zeros((4, 256), np.float32), 4, 256)
    assert e.value.status == 3
    with pytest.raises(hip_api.HipError) as e:
        hip.gemm_block_dots(Q5_K, np.zeros(176, np.uint8), np.zeros((1, 256), np.float32), 1, 1, 256)
    assert e.value.status == 3
    with pytest.raises(hip_api.HipError) as e:  # k not a multiple of 256
        hip.gemm(Q4_0, np.zeros(18 * 4, np.uint8), np.zeros((1, 128), np.float32), 1, 1, 128)
    assert e.value.status == 3


@pytest.mark.parametrize("m,n,k,amp", [(96, 5, 1024, 1.0), (300, 77, 2048, 1.0), (130, 17, 14336, 1.0), (512, 200, 4096, 1.0),
                                         (257, 65, 512, 1e-3), (64, 130, 4096, 300.0), (1, 1, 256, 1.0), (4096, 512, 4096, 1.0)])
def test_gemm_q5k_reads_f32_activations(hip, orc, m, n, k, amp):
    """The Q5_K batched kernel dots the weights with the UNQUANTIZED activations, as cera does
    (cpu.rs:1830-1854): against the exact product in f64 the error is f32-class -- far below
    what a Q8_0 round trip of x would cost (~5e-3 rms) -- at every magnitude of x, with ragged
    tiles, a split K and a lone element; and each column agrees with the Q5_K GEMV of that token."""
    _say(f"gemm Q5_K m={m} n={n} k={k} amp={amp}")
    w, _ = util.make_weights(Q5_K, m, k, seed=41 + m)
    x = (util.rng(m + n + k).standard_normal((n, k)) * amp).astype(np.float32)
    out = hip.gemm(Q5_K, w, x, m, n, k)
    rows = np.arange(m) if m <= 600 else np.unique(np.concatenate([np.arange(8), util.rng(2).integers(0, m, 48), np.arange(m - 8, m)]))
    rb = util.H.row_bytes(Q5_K, k)
    wr = np.ascontiguousarray(w.reshape(m, rb)[rows]).reshape(-1)
    exact = util.dequant_np(Q5_K, wr, rows.size, k).astype(np.float64) @ x.astype(np.float64).T
    err = np.abs(out[rows].astype(np.float64) - exact).max()
    _say(f"  max|err|={err:.3e} rms={util.rms(exact):.3e}")
    assert err <= GEMM_TOL * util.rms(exact)
    assert err <= 3e-5 * util.rms(exact), "not f32-class: the activations were rounded somewhere"
    for j in sorted({0, n // 2, n - 1}):
        y = hip.gemv(Q5_K, wr, x[j], rows.size, k)
        assert np.abs(out[rows, j] - y).max() <= 3e-5 * util.rms(exact)


def test_gemm_q5k_lets_non_finite_activations_through(hip):
    """One NaN among a token's activations makes every output of that token NaN, as the reference's
    f32 dot does (vec_dot_q5km_f32, cera/src/backend/cpu.rs:1830-1854: NaN x weight is NaN for any
    weight) and as the Q5_K GEMV of that token does; an infinity makes them non-finite; the other
    tokens of the batch are untouched."""
    m, n, k = 96, 40, 1024
    w, _ = util.make_weights(Q5_K, m, k, seed=7)
    x = util.rng(8).standard_normal((n, k)).astype(np.float32)
    clean = hip.gemm(Q5_K, w, x, m, n, k)
    bad = x.copy()
    bad[3, 517] = np.nan
    bad[29, 0] = np.inf
    bad[31, 1023] = -np.inf
    _say("gemm Q5_K with NaN / Inf activations")
    out = hip.gemm(Q5_K, w, bad, m, n, k)
    assert np.isnan(out[:, 3]).all()
    assert not np.isfinite(out[:, 29]).any() and not np.isfinite(out[:, 31]).any()
    others = [j for j in range(n) if j not in (3, 29, 31)]
    assert np.array_equal(out[:, others].view(np.uint32), clean[:, others].view(np.uint32))
    for j in (3, 29, 31):
        y = hip.gemv(Q5_K, w, bad[j], m, k)
        assert not np.isfinite(y).any()
        if j == 3:
            assert np.isnan(y).all()   # the same NaN positions as the batched kernel: all of them


def test_q5k_model_prefills_in_batches(hip, orc):
    """A model whose Q4_K tensors are Q5_K (the Q5_K_M recipe) takes the batched prefill route:
    logits and KV cache agree with the token-by-token decode of the same prompt, and with the
    oracle's per-token forward (cera's own route for a Q5_K model, llama.rs:1643)."""
    cfg = dict(synth.TINY)
    q5 = lambda name: util.H.Q5_K if synth.q4_k_m_type(name) == util.H.Q4_K else synth.q4_k_m_type(name)
    weights = synth.make_llama(cfg, seed=91, sigma=0.05, norm_jitter=0.1, type_of=q5)
    assert weights["blk.0.attn_q.weight"][0] == util.H.Q5_K and weights["blk.0.ffn_down.weight"][0] == util.H.Q6_K
    a, b = hip_api.Model(hip, cfg, weights), hip_api.Model(hip, cfg, weights)
    om = orc.Llama(cfg, weights)
    toks = [int(t) for t in util.rng(6).integers(0, cfg["vocab"], 37)]
    _say("model: Q5_K_M batched prefill 37 tokens")
    la = a.forward_prefill(toks, 0)
    for pos, t in enumerate(toks):
        lb = b.forward(t, pos)
        lo = om.forward(t, pos)
    _say(f"  batched vs per-token cos={_cos(la, lb):.8f}; vs oracle cos={_cos(la, lo):.8f}")
    assert _cos(la, lb) > 0.999 and _cos(la, lo) > 0.999
    ka, va = a.read_kv(0)
    kb, vb = b.read_kv(0)
    assert np.abs(ka - kb).max() <= 1e-4 * util.rms(kb)   # layer 0: Q5_K k-projection of identical f32 inputs
    kl, _ = a.read_kv(cfg["n_layers"] - 1)
    kr, _ = b.read_kv(cfg["n_layers"] - 1)
    assert np.abs(kl - kr).max() <= 5e-2 * util.rms(kr)
    # all-position logits through the batched head as well
    c = hip_api.Model(hip, cfg, weights)
    allg = c.forward_prefill_logits_all(toks[:12], 0)
    assert _cos(allg[-1], hip_api.Model(hip, cfg, weights).forward_prefill(toks[:12], 0)) > 0.9999
    for mdl in (a, b, c):
        mdl.close()
    om.close()


def _cos(a, b):
    a = a.astype(np.float64); b = b.astype(np.float64)
    return float(a @ b / np.sqrt((a @ a) * (b @ b)))


def test_batched_prefill_vs_oracle(hip, orc):
    cfg = dict(synth.TINY)
    weights = synth.make_llama(cfg, seed=77, sigma=0.05, norm_jitter=0.1)
    gm = hip_api.Model(hip, cfg, weights)
    om = orc.Llama(cfg, weights)
    toks = [int(t) for t in util.rng(3).integers(0, cfg["vocab"], 40)]
    _say("model: batched prefill 40 tokens")
    lg = gm.forward_prefill(toks, 0)
    lo = om.forward_prefill_batched(toks, 0)
    assert gm.seq_len == om.seq_len == 40
    _say(f"  cos={_cos(lg, lo):.8f} max|err|={np.abs(lg - lo).max():.3e} rms={util.rms(lo):.3e}")
    assert _cos(lg, lo) > 0.999
    for layer in range(cfg["n_layers"]):
        kg, vg = gm.read_kv(layer)
        ko, vo = om.kv(layer)
        # layer 0 sees identical inputs: tight; deeper layers inherit Q8_0 rounding flips
        tol = 2e-3 if layer == 0 else 5e-2
        assert np.abs(kg - ko).max() <= tol * util.rms(ko), layer
        assert np.abs(vg - vo).max() <= tol * util.rms(vo), layer
    # a second chunk on top (start_pos > 0), then decode continues from the prefilled cache
    more = [int(t) for t in util.rng(4).integers(0, cfg["vocab"], 9)]
    lg2 = gm.forward_prefill(more, 40)
    lo2 = om.forward_prefill_batched(more, 40)
    assert _cos(lg2, lo2) > 0.999
    lg3 = gm.forward(5, 49)
    lo3 = om.forward(5, 49)
    assert _cos(lg3, lo3) > 0.999
    gm.close(); om.close()


def test_prefill_equals_decode_on_gpu(hip):
    """Batched prefill and token-by-token decode of the same prompt leave the same
    KV cache and logits (to float tolerance) -- cpu.rs:5332-5425 in spirit."""
    cfg = dict(synth.TINY)
    weights = synth.make_llama(cfg, seed=78, sigma=0.05)
    a = hip_api.Model(hip, cfg, weights)
    b = hip_api.Model(hip, cfg, weights)
    toks = [int(t) for t in util.rng(5).integers(0, cfg["vocab"], 17)]
    la = a.forward_prefill(toks, 0)
    for pos, t in enumerate(toks):
        lb = b.forward(t, pos)
    assert _cos(la, lb) > 0.999
    ka, va = a.read_kv(0)
    kb, vb = b.read_kv(0)
    assert np.abs(ka - kb).max() <= 2e-3 * util.rms(kb)
    a.close(); b.close()


@pytest.mark.parametrize("rope_type,kv_f16", [(1, False), (0, False), (1, True)])
def test_prefill_where_the_norm_adds_split_k_partial_sums(hip, orc, rope_type, kv_f16):
    """Projections whose K is split (2048-wide rows, few row tiles) in a pass of 128 tokens or more: the O
    and down projections leave their partial sums to the row norm that follows (and the last layer's down
    projection to the reduction kernel), Q | K and V theirs to the RoPE / append kernel (both pair orders,
    f32 and f16 cache).  Logits and both layers' K/V rows track the oracle's batched prefill, and a decode
    step continues from the cache."""
    cfg = dict(synth.TINY, hidden=2048, ffn=2048, n_heads=16, n_kv_heads=4, head_dim=128, max_seq_len=192, rope_type=rope_type)
    weights = synth.make_llama(cfg, seed=81, sigma=0.03, norm_jitter=0.1)
    gm = hip_api.Model(hip, cfg, weights)
    om = orc.Llama(cfg, weights)
    if kv_f16:
        gm.configure_kv(True); om.set_kv_f16(True)
    toks = [int(t) for t in util.rng(12).integers(0, cfg["vocab"], 130)]
    _say("model: 130-token prefill, hidden 2048 (split-K O and down projections)")
    lg = gm.forward_prefill(toks, 0)
    lo = om.forward_prefill_batched(toks, 0)
    _say(f"  cos={_cos(lg, lo):.8f} max|err|={np.abs(lg - lo).max():.3e} rms={util.rms(lo):.3e}")
    assert _cos(lg, lo) > 0.999
    for layer in range(cfg["n_layers"]):
        kg, vg = gm.read_kv(layer)
        ko, vo = om.kv(layer)
        tol = 2e-3 if layer == 0 else 5e-2
        assert np.abs(kg - ko).max() <= tol * util.rms(ko), layer
        assert np.abs(vg - vo).max() <= tol * util.rms(vo), layer
    lg2 = gm.forward(7, 130)
    lo2 = om.forward(7, 130)
    assert _cos(lg2, lo2) > 0.999
    gm.close(); om.close()


@pytest.mark.parametrize("head_dim,n_heads,n_kv_heads", [(8, 32, 8), (40, 32, 2), (64, 4, 4), (256, 3, 1)])
@pytest.mark.parametrize("rope_type,kv_f16", [(1, False), (0, False), (1, True), (0, True)])
def test_prefill_rotates_heads_of_every_size(hip, orc, head_dim, n_heads, n_kv_heads, rope_type, kv_f16):
    """Rotation and append over heads that do not fill a workgroup's threads evenly, both pair orders and cache types, from position 0
    and from inside a sequence.  Layer 0's rows are one product away from the oracle's: its tolerance, as above."""
    cfg = dict(synth.TINY, n_layers=1, hidden=512, n_heads=n_heads, n_kv_heads=n_kv_heads, head_dim=head_dim, max_seq_len=96, rope_type=rope_type)
    weights = synth.make_llama(cfg, seed=83, sigma=0.03, norm_jitter=0.1)
    gm = hip_api.Model(hip, cfg, weights)
    om = orc.Llama(cfg, weights)
    if kv_f16:
        gm.configure_kv(True); om.set_kv_f16(True)
    toks = [int(t) for t in util.rng(head_dim).integers(0, cfg["vocab"], 81)]
    _say(f"model: heads of {head_dim}, {n_heads} / {n_kv_heads}, rope {rope_type}, f16 cache {kv_f16}")
    for first, last in ((0, 10), (10, 81)):
        gm.forward_prefill(toks[first:last], first)
        om.forward_prefill_batched(toks[first:last], first)
    (kg, vg), (ko, vo) = gm.read_kv(0), om.kv(0)
    assert np.abs(kg - ko).max() <= 2e-3 * util.rms(ko)
    assert np.abs(vg - vo).max() <= 2e-3 * util.rms(vo)
    gm.close(); om.close()


@pytest.mark.parametrize("head_dim,n_heads,n_kv_heads,hidden,cuts", [(8, 64, 64, 512, (42, 43)), (40, 32, 32, 512, (85, 86)), (64, 32, 32, 512, (1, 97)),
                                                                     (256, 16, 16, 512, (86, 85)), (64, 4, 1, 2048, (256, 257)), (64, 4, 1, 16384, (32, 33))])
@pytest.mark.parametrize("rope_type,kv_f16", [(1, False), (0, True)])
def test_prefill_on_both_sides_of_a_round_of_the_chip(hip, orc, head_dim, n_heads, n_kv_heads, hidden, cuts, rope_type, kv_f16):
    """Rotation by pairs and by quads, embedding by one element and by four: the launches in passes of up to, and of more than, the
    8192 wavefronts that 256 CUs hold.  Tolerance: as above, and in an f16 cache a step of the value on top, 2^-10 of it at most: both
    sides round to f16, and a difference of any size may put them on neighbours."""
    n = sum(cuts)
    cfg = dict(synth.TINY, n_layers=1, hidden=hidden, ffn=256, n_heads=n_heads, n_kv_heads=n_kv_heads, head_dim=head_dim, max_seq_len=n, rope_type=rope_type)
    weights = synth.make_llama(cfg, seed=89, sigma=0.03, norm_jitter=0.1)
    gm = hip_api.Model(hip, cfg, weights)
    om = orc.Llama(cfg, weights)
    if kv_f16:
        gm.configure_kv(True); om.set_kv_f16(True)
    toks = [int(t) for t in util.rng(head_dim).integers(0, cfg["vocab"], n)]
    _say(f"model: heads of {head_dim}, {n_heads} / {n_kv_heads}, hidden {hidden}, rope {rope_type}, f16 cache {kv_f16}, passes of {cuts}")
    for first, last in ((0, cuts[0]), (cuts[0], n)):
        gm.forward_prefill(toks[first:last], first)
        om.forward_prefill_batched(toks[first:last], first)
    (kg, vg), (ko, vo) = gm.read_kv(0), om.kv(0)
    for got, want in ((kg, ko), (vg, vo)):
        assert (np.abs(got - want) <= 2e-3 * util.rms(want) + (np.abs(want) * 2.0 ** -10 if kv_f16 else 0)).all()
    gm.close(); om.close()


# a pass of a few tokens: (config, make_llama's arguments, biases, QK norm, f16 cache)
FEW_MODELS = {
    "q4_k_m": (dict(), dict(), False, False, False),                                        # Q | K and a Q6_K V in one launch
    "q4_k_m_neox_f16": (dict(rope_type=0), dict(), False, False, True),
    "q4_k": (dict(), dict(type_of=lambda name: Q4_K), False, False, False),                 # one joint Q | K | V
    "q6_k_f16": (dict(), dict(type_of=lambda name: Q6_K), False, False, True),
    "q4_k_m_bias": (dict(rope_type=0), dict(), True, False, False),                         # RoPE cannot add the sums up
    "q4_k_qknorm": (dict(rope_type=0), dict(type_of=lambda name: Q4_K), False, True, False),
    "granite_scalars": (dict(embed_scale=12.0, residual_scale=0.22, attn_scale=0.0078125, logit_scale=8.0), dict(), False, False, False),
    "q5_k_m": (dict(), dict(type_of=lambda name: Q5_K if synth.q4_k_m_type(name) == Q4_K else synth.q4_k_m_type(name)), False, False, False),
    "q8_0": (dict(), dict(type_of=lambda name: Q8_0), False, False, False),                 # only the norm of a few rows is another
}


@pytest.mark.parametrize("name", list(FEW_MODELS))
def test_passes_of_a_few_tokens_vs_oracle(hip, orc, name):
    """Portions of 2 to 49 tokens of a 2048-wide model, one behind the other, against the oracle fed the same portions:
    joint Q | K (| V) outputs in their segments, sums over slices of K left to RoPE and to the row norm with the residual
    and its scale, both caches, and the same behind biases and QK norms, which keep RoPE from adding up.  The first layer's
    cache rows have only one product behind them.  Beyond it codes flip: a difference d in front of a rounding to steps of s
    leaves sqrt(d s) behind it, so last bits grow to the rounding's own noise within a layer.  A step is 2.3 / 127 of a
    block's rms, two routes' noise 2 / 12 of its square per rounded input, four of them lie in front of the second layer's
    rows (1.5 % of the rms together), and the largest of their 1e5 differences is 4.6 times that: 7e-2."""
    over, mk, bias, qk_norm, kv_f16 = FEW_MODELS[name]
    cfg = dict(synth.TINY, hidden=2048, ffn=2304, n_heads=16, n_kv_heads=4, head_dim=128, max_seq_len=256, **over)
    weights = synth.make_llama(cfg, seed=83, sigma=0.03, norm_jitter=0.1, **mk)
    r = util.rng(8)
    for i in range(cfg["n_layers"]):
        for part, rows in (("q", 2048), ("k", 512), ("v", 512)):
            if bias:
                weights[f"blk.{i}.attn_{part}.bias"] = (r.standard_normal(rows) * 0.5).astype(np.float32)
            if qk_norm and part != "v":
                weights[f"blk.{i}.attn_{part}_norm.weight"] = (1.0 + 0.3 * r.standard_normal(128)).astype(np.float32)
    gm, om = hip_api.Model(hip, cfg, weights), orc.Llama(cfg, weights)
    if kv_f16:
        gm.configure_kv(True); om.set_kv_f16(True)
    at = 0
    for n in (5, 17) if name == "q5_k_m" else (5, 48, 3, 33, 16, 17, 2, 32, 49):
        toks = [int(t) for t in r.integers(0, cfg["vocab"], n)]
        if n == 33:   # all positions' logits: the last row is the oracle's, the others what a shorter portion ends in
            got = gm.forward_prefill_logits_all(toks, at)
            gm.truncate_kv(at)
            short = gm.forward_prefill(toks[:20], at)
            gm.truncate_kv(at)
            lg = gm.forward_prefill(toks, at)
            assert _cos(got[19], short) > 0.999 and _cos(got[-1], lg) > 0.999
        else:
            lg = gm.forward_prefill(toks, at)
        # (the oracle has no batched Q5_K)
        lo = (om.forward_prefill_per_token if name == "q5_k_m" else om.forward_prefill_batched)(toks, at)
        _say(f"{name}: {n} tokens behind {at}: cos {_cos(lg, lo):.8f} max|err| {np.abs(lg - lo).max():.3e} of rms {util.rms(lo):.3e}")
        assert _cos(lg, lo) > 0.999, (n, at)
        at += n
    for layer in range(cfg["n_layers"]):
        for got, want in zip(gm.read_kv(layer), om.kv(layer)):
            err = np.abs(got - want).max() / util.rms(want)
            _say(f"  layer {layer}: {err:.2e}")
            # (an f16 cache: a value next to a rounding boundary is 2^-11 of itself off, of six times the rms at most)
            assert err <= (7e-2 if layer else 3e-3 if kv_f16 else 2e-3), layer
    gm.close(); om.close()


@pytest.mark.parametrize("n", [12, 49, 70, 200])
def test_prefill_of_a_model_all_in_q6_k(hip, orc, n):
    """Q6_K gate and up in front of a Q6_K down projection: the f16 form of the normed activations, which gate and up
    leave behind, is not the down projection's input.  A pass of 64-token tiles, and of the records of more tokens."""
    cfg = dict(synth.TINY, max_seq_len=256)
    weights = synth.make_llama(cfg, seed=84, sigma=0.05, norm_jitter=0.1, type_of=lambda name: Q6_K)
    gm, om = hip_api.Model(hip, cfg, weights), orc.Llama(cfg, weights)
    toks = [int(t) for t in util.rng(n).integers(0, cfg["vocab"], n)]
    lg, lo = gm.forward_prefill(toks, 0), om.forward_prefill_batched(toks, 0)
    _say(f"q6_k model, {n} tokens: cos {_cos(lg, lo):.8f}")
    assert _cos(lg, lo) > 0.999
    gm.close(); om.close()


@pytest.mark.parametrize("nh,nkv,start,n", [(32, 8, 0, 512), (8, 2, 0, 40), (8, 8, 300, 100), (16, 2, 1000, 33),
                                             (4, 1, 0, 16), (32, 8, 4000, 96), (32, 8, 2048, 2048)])
def test_attn_prefill_batch_vs_oracle(hip, orc, nh, nkv, start, n):
    """Causal attention of a batch of queries (the tiled MFMA kernel) against the oracle's
    decode_attention evaluated query by query: query i sees positions 0 .. start + i."""
    hd = 128
    _say(f"attn_prefill nh={nh} nkv={nkv} start={start} n={n}")
    r = util.rng(7 * n + start)
    L = start + n
    q = r.standard_normal((n, nh * hd), dtype=np.float32)
    k = r.standard_normal(L * nkv * hd, dtype=np.float32)
    v = r.standard_normal(L * nkv * hd, dtype=np.float32)
    scale = 1.0 / np.sqrt(hd)
    out = hip.attn_prefill(q, k, v, nh, nkv, hd, start, n, scale)
    picks = sorted(set([0, 1, 15, 16, 31, 32, n // 2, n - 2, n - 1]) & set(range(n)))
    for i in picks:
        Li = start + i + 1
        ref = orc.decode_attention(q[i], k[:Li * nkv * hd], v[:Li * nkv * hd], nh, nkv, hd, scale, Li)
        err = np.abs(out[i].astype(np.float64) - ref).max()
        assert err <= 2e-3 * util.rms(ref), (i, err, util.rms(ref))
    assert np.isfinite(out).all()


@pytest.mark.parametrize("kv_f16", [False, True])
@pytest.mark.parametrize("nh,nkv,hd,start,n", [(32, 8, 128, 16, 16), (8, 1, 128, 5000, 20), (6, 2, 64, 2079, 33), (32, 8, 128, 900, 12), (8, 1, 64, 17, 8),
                                               (64, 8, 128, 3000, 15)])
def test_attn_of_few_queries_in_parts(hip, orc, nh, nkv, hd, start, n, kv_f16):
    """16 and more queries whose blocks leave the chip idle: parts of one tile of 32 keys, the most parts that there are (64, two
    rounds of the merge's lanes), a last part and a last block that are not whole; and 8 to 15 queries, which share the keys' rows.
    Bound as for the accuracy of the split products below."""
    _say(f"attn few queries nh={nh} nkv={nkv} hd={hd} start={start} n={n} f16={kv_f16}")
    r = util.rng(n + start)
    L = start + n
    q = r.standard_normal((n, nh * hd), dtype=np.float32)
    k, v = (r.standard_normal(L * nkv * hd, dtype=np.float32) for _ in range(2))
    if kv_f16:
        k, v = (x.astype(np.float16).astype(np.float32) for x in (k, v))
    scale = 1.0 / np.sqrt(hd)
    out = (hip.attn_f16kv if kv_f16 else hip.attn_prefill)(q, k, v, nh, nkv, hd, start, n, scale)
    for i in sorted({0, n // 2, n - 1}):
        Li = start + i + 1
        ref = orc.decode_attention(q[i], k[:Li * nkv * hd], v[:Li * nkv * hd], nh, nkv, hd, scale, Li)
        assert np.abs(out[i].astype(np.float64) - ref).max() <= 5e-5 * util.rms(ref), i


@pytest.mark.parametrize("case", ["plain", "wide_range", "sink"])
def test_attn_prefill_split_f16_keeps_f32_accuracy(hip, orc, case):
    """The batch kernel multiplies on the f16 matrix cores with every operand split into an f16
    high and low part.  Its error against the f32 reference must stay at f32 level (far inside
    the 2e-3 bar a plain f16 product would only just meet), also when the operands span many
    binades and when the weights are one dominant key (an attention sink) plus thousands of
    keys at 1e-4 of it, where f16 alone would round the small weights coarsely."""
    nh, nkv, hd, start, n = 8, 2, 128, 3000, 64
    _say(f"attn_prefill split-f16 accuracy case={case}")
    r = util.rng(1234)
    L = start + n
    q = r.standard_normal((n, nh * hd), dtype=np.float32)
    k = r.standard_normal((L, nkv * hd), dtype=np.float32)
    v = r.standard_normal((L, nkv * hd), dtype=np.float32)
    if case == "wide_range":
        # per-dimension magnitudes from 2^-12 to 2^6: f16 subnormal low parts and large values
        mag = np.exp2(r.integers(-12, 7, hd)).astype(np.float32)
        k *= np.tile(mag, nkv); q /= np.tile(mag, nh); v *= np.tile(mag[::-1], nkv)
    if case == "sink":
        # key 0 lines up with every query: one weight of 1 against thousands near exp(-9)
        k *= 0.05
        k[0] = 0.0
        k[0, ::hd] = 60.0          # dim 0 of every KV head
        q[:, ::hd] = np.abs(q[:, ::hd]) + 2.0
    scale = 1.0 / np.sqrt(hd)
    out = hip.attn_prefill(q, k.reshape(-1), v.reshape(-1), nh, nkv, hd, start, n, scale)
    worst = 0.0
    for i in (0, 31, 32, n - 1):
        Li = start + i + 1
        ref = orc.decode_attention(q[i], k[:Li].reshape(-1), v[:Li].reshape(-1), nh, nkv, hd, scale, Li)
        worst = max(worst, np.abs(out[i].astype(np.float64) - ref).max() / util.rms(ref))
    _say(f"  max|err| / rms = {worst:.3e}")
    assert worst <= 5e-5


@pytest.mark.parametrize("kv_f16", [False, True])
@pytest.mark.parametrize("nh,nkv,start,n", [(32, 8, 0, 200), (8, 2, 300, 40), (4, 4, 1000, 33)])
def test_attn_prefill_batch_head_dim_64(hip, orc, kv_f16, nh, nkv, start, n):
    hd = 64
    _say(f"attn_prefill hd=64 nh={nh} nkv={nkv} start={start} n={n} f16={kv_f16}")
    r = util.rng(13 * n + start)
    L = start + n
    q = r.standard_normal((n, nh * hd), dtype=np.float32)
    k = r.standard_normal(L * nkv * hd, dtype=np.float32)
    v = r.standard_normal(L * nkv * hd, dtype=np.float32)
    scale = 1.0 / np.sqrt(hd)
    if kv_f16:
        out = hip.attn_f16kv(q, k, v, nh, nkv, hd, start, n, scale)
        k = k.astype(np.float16).astype(np.float32); v = v.astype(np.float16).astype(np.float32)
    else:
        out = hip.attn_prefill(q, k, v, nh, nkv, hd, start, n, scale)
    for i in sorted(set([0, 1, 31, 32, n // 2, n - 1]) & set(range(n))):
        Li = start + i + 1
        ref = orc.decode_attention(q[i], k[:Li * nkv * hd], v[:Li * nkv * hd], nh, nkv, hd, scale, Li)
        err = np.abs(out[i].astype(np.float64) - ref).max()
        assert err <= 2e-3 * util.rms(ref), (i, err, util.rms(ref))


@pytest.mark.parametrize("nh,nkv,hd,kv_f16,start,n", [(8, 2, 128, False, 1500, 290), (3, 1, 128, False, 0, 961), (14, 2, 128, True, 900, 481),
                                                       (8, 1, 128, False, 31, 970), (2, 2, 64, True, 1200, 353), (6, 3, 64, False, 3001, 161),
                                                       (16, 8, 128, False, 1500, 290)])
def test_attn_prefill_of_many_queries(hip, orc, nh, nkv, hd, kv_f16, start, n):
    """Batches large enough that the cache's tiles are split once and read as records (and one shape, two heads a group, that
    keeps the other kernel): blocks that end inside a tile of 32 keys, last blocks of one query and of all 32, each group size's
    way of dividing a record.  A value that is not finite at a later position must not come through to a block of queries
    before it, though its tile is read there; the bound is that of the smaller batches."""
    _say(f"attn_prefill many nh={nh} nkv={nkv} hd={hd} start={start} n={n} f16={kv_f16}")
    r = util.rng(17 * n + start)
    L = start + n
    q = r.standard_normal((n, nh * hd), dtype=np.float32)
    k = r.standard_normal((L, nkv * hd), dtype=np.float32)
    v = r.standard_normal((L, nkv * hd), dtype=np.float32)
    bad = start + 64   # the first key behind the first two blocks of queries
    v[bad] = np.nan
    if kv_f16:
        k = k.astype(np.float16).astype(np.float32); v = v.astype(np.float16).astype(np.float32)
    scale = 1.0 / np.sqrt(hd)
    fn = hip.attn_f16kv if kv_f16 else hip.attn_prefill
    picks = sorted({0, 31, 32, 63, 64, n // 2, n - 2, n - 1})
    for poison in (True, False):
        if not poison:
            v[bad] = 0.5
        out = fn(q, k.reshape(-1), v.reshape(-1), nh, nkv, hd, start, n, scale)
        for i in picks:
            if poison and i >= 64:
                continue
            Li = start + i + 1
            ref = orc.decode_attention(q[i], k[:Li].reshape(-1), v[:Li].reshape(-1), nh, nkv, hd, scale, Li)
            err = np.abs(out[i].astype(np.float64) - ref).max()
            assert err <= 2e-3 * util.rms(ref), (poison, i, err, util.rms(ref))
        assert np.isfinite(out[:64] if poison else out).all()


def test_attn_prefill_without_room_for_records():
    """The split tiles of the cache are a workspace that the pass can do without: where it cannot be had (here by a limit
    that the inputs fit and the records do not), the kernel without it runs, with the same products in the same order."""
    nh, nkv, hd, start, n = 8, 2, 128, 1500, 290
    r = util.rng(3)
    L = start + n
    q = r.standard_normal((n, nh * hd), dtype=np.float32)
    k, v = (r.standard_normal(L * nkv * hd, dtype=np.float32) for _ in range(2))
    out = []
    for limit in (0, 5 << 19):
        ctx = hip_api.Context(0)
        ctx.set_workspace_limit(limit)
        _say(f"attn_prefill many, workspace limit {limit}")
        out.append(ctx.attn_prefill(q, k, v, nh, nkv, hd, start, n, 1.0 / np.sqrt(hd)))
        ctx.close()
    assert np.array_equal(out[0].view(np.uint32), out[1].view(np.uint32))


def test_records_of_a_growing_context_take_their_room_once():
    """Passes further and further into a context split more and more tiles: the room for them is that of the whole cache from
    the first pass on, so that no later one stops to allocate."""
    cfg = dict(synth.TINY, hidden=512, ffn=512, n_heads=24, n_kv_heads=8, head_dim=128, n_layers=1, max_seq_len=4096)
    ctx = hip_api.Context(0)
    m = hip_api.Model(ctx, cfg, synth.make_llama(cfg, seed=5, sigma=0.05))
    toks = [int(t) for t in util.rng(6).integers(0, cfg["vocab"], 4000)]
    free = []
    for at in range(0, 4000, 1000):
        m.forward_prefill(toks[at:at + 1000], at)
        free.append(util.free_device_bytes())
        _say(f"prefill of 1000 tokens behind {at}: {free[-1]} bytes free")
    m.close()
    ctx.close()
    assert len(set(free)) == 1


def test_prefill_longer_than_one_pass(hip, orc):
    """A prompt beyond the 2048-token pass size is cut into passes; logits and the cache rows on
    both sides of the cut track the oracle's single batched prefill."""
    cfg = dict(synth.TINY, max_seq_len=2200)
    weights = synth.make_llama(cfg, seed=79, sigma=0.05, norm_jitter=0.1)
    gm = hip_api.Model(hip, cfg, weights)
    om = orc.Llama(cfg, weights)
    toks = [int(t) for t in util.rng(9).integers(0, cfg["vocab"], 2100)]
    _say("model: prefill 2100 tokens (two passes)")
    lg = gm.forward_prefill(toks, 0)
    lo = om.forward_prefill_batched(toks, 0)
    assert gm.seq_len == om.seq_len == 2100
    assert _cos(lg, lo) > 0.999
    kvd = cfg["n_kv_heads"] * cfg["head_dim"]
    kg, vg = gm.read_kv(0)
    ko, vo = om.kv(0)
    rows = slice(2040 * kvd, 2060 * kvd)
    assert np.abs(kg[rows] - ko[rows]).max() <= 2e-3 * util.rms(ko[rows])
    assert np.abs(vg[rows] - vo[rows]).max() <= 2e-3 * util.rms(vo[rows])
    lg2, lo2 = gm.forward(3, 2100), om.forward(3, 2100)
    assert _cos(lg2, lo2) > 0.999
    gm.close(); om.close()


@pytest.mark.parametrize("n", [5, 40])
def test_batched_prefill_when_k_is_not_a_multiple_of_256(hip, orc, n):
    """Small models' hidden sizes (896, 1536 ...) have no int8-GEMM form; their Q4_0 / Q8_0 matrices
    still take a batch through the multi-token GEMV (8 tokens per weight pass) instead of one decode
    step per token.  hidden 288, ffn 480: every K is a multiple of 32 only."""
    cfg = dict(synth.TINY, hidden=288, ffn=480, n_heads=4, n_kv_heads=2, head_dim=64)
    type_of = lambda name: Q8_0 if ("attn_v" in name or "ffn_down" in name or "token_embd" in name) else Q4_0
    weights = synth.make_llama(cfg, seed=83, sigma=0.05, type_of=type_of, norm_jitter=0.1)
    gm = hip_api.Model(hip, cfg, weights)
    om = orc.Llama(cfg, weights)
    toks = [int(t) for t in util.rng(19 + n).integers(0, cfg["vocab"], n)]
    _say(f"model: hidden 288, batched prefill of {n} tokens over Q4_0 / Q8_0")
    lg = gm.forward_prefill(toks, 0)
    lo = om.forward_prefill_per_token(toks, 0)
    assert gm.seq_len == om.seq_len == n
    assert _cos(lg, lo) > 0.999
    kg, vg = gm.read_kv(1)
    ko, vo = om.kv(1)
    assert np.abs(kg - ko).max() <= 5e-2 * util.rms(ko) and np.abs(vg - vo).max() <= 5e-2 * util.rms(vo)
    rows = gm.forward_prefill_logits_all([3, 4, 5], n)
    for i, t in enumerate([3, 4, 5]):
        assert _cos(rows[i], om.forward(t, n + i)) > 0.999, i
    gm.close(); om.close()


# ---- config 3 at the shapes the benchmark times ---------------------------------------------------
def _row_sample_check(hip, orc, dtype, w, m, k, x, n, rows):
    out = hip.gemm(dtype, w, x, m, n, k)
    rb = util.H.row_bytes(dtype, k)
    wr = np.ascontiguousarray(w.reshape(m, rb)[rows]).reshape(-1)
    ref = _oracle_gemm(orc, dtype, wr, x, rows.size, n, k)
    err = np.abs(out[rows].astype(np.float64) - ref).max()
    assert err <= GEMM_TOL * util.rms(ref), (err, util.rms(ref))
    return out


@pytest.mark.parametrize("dtype,m,k", [(Q4_K, 14336, 4096), (Q4_K, 6144, 4096)])
@pytest.mark.parametrize("n", [128, 512, 2048])
def test_gemm_config3_gate_and_qkv_shapes(hip, orc, dtype, m, k, n):
    """The gate/up projection (the shape the benchmark times) and the fused QKV height."""
    _say(f"gemm config 3 {util.NAMES[dtype]} m={m} n={n} k={k}")
    w, _ = util.make_weights(dtype, m, k, seed=11)
    x = util.rng(n + 1).standard_normal((n, k)).astype(np.float32)
    rows = np.unique(np.concatenate([np.arange(8), util.rng(2).integers(0, m, 48), np.arange(m - 8, m)]))
    _row_sample_check(hip, orc, dtype, w, m, k, x, n, rows)


@pytest.fixture(scope="module")
def head_q6k():
    m, k = 128256, 4096
    w, _ = util.make_weights(Q6_K, m, k, seed=12)
    return w, m, k


@pytest.mark.parametrize("n", [128, 512, 2048])
def test_gemm_config3_vocabulary_head(hip, orc, head_q6k, n):
    """The Q6_K output head 128256 x 4096 (the all-position logits GEMM), row-sampled."""
    w, m, k = head_q6k
    _say(f"gemm config 3 Q6_K head m={m} n={n} k={k}")
    x = util.rng(n + 2).standard_normal((n, k)).astype(np.float32)
    rows = np.unique(np.concatenate([np.arange(4), util.rng(3).integers(0, m, 40), np.arange(m - 4, m)]))
    _row_sample_check(hip, orc, Q6_K, w, m, k, x, n, rows)


@pytest.mark.parametrize("n", [128, 512, 2048])
def test_gemm_swiglu_at_ffn_shape_against_the_oracle(hip, orc, n):
    """The prefill pass's fused gate | up | SwiGLU | Q8_0 launch at 14336 x 4096, against the
    oracle's own chain gemm_preq -> silu_mul_inplace -> quantize_columns (transformer.rs:710-788,
    cpu.rs:2570-2575, transformer.rs:865-946) on a sample of 32-row quantization blocks.  The GEMM
    outputs agree with the oracle's to the float bar only, so a value that sits on a rounding
    boundary may land one int8 step away and a block maximum may round to the neighbouring f16
    scale: the dequantized result must meet the oracle's SwiGLU output within one quantization
    step, codes may differ by at most one step and only rarely, scales by at most one f16 ulp."""
    m, k = 14336, 4096
    _say(f"gemm_swiglu 14336x4096 vs oracle n={n}")
    wg, _ = util.make_weights(Q4_K, m, k, seed=51)
    wu, _ = util.make_weights(Q4_K, m, k, seed=52)
    x = util.rng(53 + n).standard_normal((n, k)).astype(np.float32)
    q, sc, fused = hip.gemm_swiglu(Q4_K, wg, wu, m, x, n, k)
    assert fused == (n >= 512), "small batches take the pair + SwiGLU kernels, large ones the fused launch"
    blocks = np.unique(np.concatenate([[0, 1, m // 32 - 1], util.rng(4).integers(0, m // 32, 5)]))
    rows = (blocks[:, None] * 32 + np.arange(32)[None, :]).reshape(-1)
    rb = util.H.row_bytes(Q4_K, k)
    g = _oracle_gemm(orc, Q4_K, np.ascontiguousarray(wg.reshape(m, rb)[rows]).reshape(-1), x, rows.size, n, k)
    u = _oracle_gemm(orc, Q4_K, np.ascontiguousarray(wu.reshape(m, rb)[rows]).reshape(-1), x, rows.size, n, k)
    h = orc.silu_mul(np.ascontiguousarray(g.T).reshape(-1), np.ascontiguousarray(u.T).reshape(-1)).reshape(n, rows.size)
    rs, rq = orc.quantize_q8_0(h.reshape(-1))
    rs, rq = rs.reshape(n, blocks.size), rq.reshape(n, rows.size)
    gq, gs = q[:, rows], sc[:, blocks]
    dq = np.abs(gq.astype(np.int32) - rq.astype(np.int32))
    assert dq.max() <= 1, int(dq.max())
    assert np.count_nonzero(dq) <= 0.02 * dq.size, np.count_nonzero(dq) / dq.size
    ulp = np.abs(gs.astype(np.float16).view(np.int16).astype(np.int32) - rs.astype(np.float16).view(np.int16).astype(np.int32))
    assert np.array_equal(gs, gs.astype(np.float16).astype(np.float32)) and ulp.max() <= 1
    deq = gq.astype(np.float32).reshape(n, blocks.size, 32) * gs[:, :, None]
    step = rs[:, :, None]
    assert (np.abs(deq - h.reshape(n, blocks.size, 32)) <= 1.01 * step + 1e-9).all()


# ---- the GEMM's integer block dots, and the route an x86 host really runs ------------------------
@pytest.mark.parametrize("dtype", util.INT8_TYPES)
@pytest.mark.parametrize("m,n,k", [(130, 70, 512), (64, 33, 1024), (9, 1, 256), (200, 5, 2048)])
def test_gemm_integer_block_dots_bit_exact(hip, orc, dtype, m, n, k):
    """Every (row, token, block) integer dot the matrix cores produce inside the prefill GEMM equals
    the brute-force integer reference (the quantities of simd.rs:6609-6629): int32 tiles of the
    int8 MFMA for Q4_0 / Q8_0 / Q4_1 / Q4_K, and for Q6_K the f32 results of the f16 MFMA, one per
    16-element scale group, which must be exact integers sum (q - 32) a.  Products of Q4_0, Q8_0 and, with many
    tokens, Q6_K run other kernels: test_block_results_are_whole_numbers reads theirs from the outputs."""
    _say(f"gemm block dots {util.NAMES[dtype]} m={m} n={n} k={k}")
    w, _ = util.make_weights(dtype, m, k, seed=dtype + m)
    x = util.rng(n + k).standard_normal((n, k)).astype(np.float32) * np.float32(3.0)
    dots, out = hip.gemm_block_dots(dtype, w, x, m, n, k)
    for j in range(n):
        _, xq = orc.quantize_q8_0(x[j])
        ref, asums = orc.block_dots(dtype, w, m, k, xq)
        if dtype == Q6_K:
            want = (ref - 32 * asums[None, :]).astype(np.float32)     # the kernel recentres the codes
            assert np.array_equal(dots[:, j, :], want), j
        else:
            assert np.array_equal(dots[:, j, :], ref), j
    ref_out = _oracle_gemm(orc, dtype, w, x, m, n, k)
    assert np.abs(out.astype(np.float64) - ref_out).max() <= GEMM_TOL * util.rms(ref_out)


@pytest.mark.parametrize("dtype,m,k,n", [(Q4_K, 14336, 4096, 512), (Q4_K, 4096, 4096, 128), (Q4_K, 6144, 4096, 2048),
                                         (Q4_0, 4096, 4096, 512)])
def test_gemm_against_the_x86_repacked_route(hip, orc, dtype, m, k, n):
    """cera on an x86 host multiplies repacked Q4_0 / Q4_K weights with the 8-row-interleaved
    kernels (gemm_q4_k_8x8_q8_0, cera/src/backend/simd.rs:5392-5518), not the standard-layout
    ones: the HIP GEMM meets the float bar against that route too (whole 8-row super-rows sampled)."""
    _say(f"gemm vs x86 8x8 route {util.NAMES[dtype]} m={m} n={n} k={k}")
    w, _ = util.make_weights(dtype, m, k, seed=21)
    x = util.rng(n + 9).standard_normal((n, k)).astype(np.float32)
    out = hip.gemm(dtype, w, x, m, n, k)
    srs = np.unique(np.concatenate([[0, m // 8 - 1], util.rng(6).integers(0, m // 8, 6)]))
    rows = (srs[:, None] * 8 + np.arange(8)[None, :]).reshape(-1)
    rb = util.H.row_bytes(dtype, k)
    wr = np.ascontiguousarray(w.reshape(m, rb)[rows]).reshape(-1)
    bs = np.empty((n, k // 32), np.float32); bq = np.empty((n, k), np.int8)
    for j in range(n):
        bs[j], bq[j] = orc.quantize_q8_0(x[j])
    ref = orc.gemm_preq_x86(dtype, wr, bs, bq, rows.size, n, k)
    assert np.abs(out[rows].astype(np.float64) - ref).max() <= GEMM_TOL * util.rms(ref)
