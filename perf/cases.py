"""The timed work: what a serving program has this framework do, through its public model calls.

A case is one call on a loaded model that already holds ``start`` tokens: one decoded token, a few drafted tokens
verified together, a chat turn, a prompt.  The model families are the llama on block-quantized weights and the two
bf16 designs read from a config.json (Nafevik, Fidinex), at the layer sizes the benchmark uses; models are cut to a few
layers, since layers repeat, and keep the vocabulary of 32000 of the benchmark's design runs.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from cera_amd import hip_api as A

VOCAB = 32000
RANK, ROT, STREAMS, LATENT_EVERY = 512, 64, 4, 4      # Fidinex: latent size, rotated entries, residual streams, latent layers
CHUNK, TAPS = 2048, 4                                 # Nafevik: positions of an attention chunk, convolution taps
ROPE_BASE, EPS = 500000.0, 1e-5
SIZES = {"4096": dict(width=4096, ff=14336, heads=32, kv_heads=8, dim=128), "3072": dict(width=3072, ff=8192, heads=24, kv_heads=8, dim=128),
         "2048": dict(width=2048, ff=8192, heads=32, kv_heads=8, dim=64)}
# block types of a llama's (embedding and most matrices, value and down projections, head)
MIXES = {"q4_k_m": (A.Q4_K, A.Q6_K, A.Q6_K), "q5_k_m": (A.Q5_K, A.Q6_K, A.Q6_K), "q4_0": (A.Q4_0, A.Q4_0, A.Q6_K), "q8_0": (A.Q8_0, A.Q8_0, A.Q6_K)}


def _case(family, size, layers, start, n, **more):
    return {"family": family, "layers": layers, **SIZES[size], "start": start, "n": n, "all": False, **more}


def listed():
    return [
        # a chat reply being written: the flagship type mix, some hundred tokens in
        {"name": "llama_decode", **_case("llama", "4096", 4, 640, 1, quant="q4_k_m", kv_f16=False)},
        # the first words of a reply of a small model: the smallest call, nothing but launches and weights
        {"name": "llama_decode_small", **_case("llama", "2048", 4, 37, 1, quant="q4_0", kv_f16=False)},
        # a question about a long document held in a half-precision cache
        {"name": "llama_decode_long", **_case("llama", "4096", 2, 15001, 1, quant="q8_0", kv_f16=True)},
        # one round of speculative decoding: the drafted tokens verified at once
        {"name": "llama_verify", **_case("llama", "4096", 2, 900, 5, quant="q4_k_m", kv_f16=False, all=True)},
        # a short user turn inside a chat
        {"name": "llama_turn", **_case("llama", "4096", 2, 700, 45, quant="q4_k_m", kv_f16=False)},
        # the benchmark's prompt
        {"name": "llama_prefill", **_case("llama", "4096", 2, 0, 512, quant="q4_k_m", kv_f16=False)},
        # a long prompt, one full pass of it in the middle
        {"name": "llama_prefill_long", **_case("llama", "4096", 2, 4096, 2048, quant="q4_k_m", kv_f16=False)},
        # a prompt of uneven length on 8-bit weights
        {"name": "llama_prefill_q8_0", **_case("llama", "3072", 2, 0, 1001, quant="q8_0", kv_f16=False)},
        # the bf16 designs: a token deep in the first chunk, and a prompt of uneven length
        {"name": "nafevik_decode", **_case("nafevik", "3072", 4, 1900, 1)},
        {"name": "nafevik_prefill", **_case("nafevik", "4096", 2, 0, 1900)},
        {"name": "fidinex_decode", **_case("fidinex", "2048", 4, 540, 1)},
        {"name": "fidinex_prefill", **_case("fidinex", "3072", 4, 777, 2048)},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    family = rng.choice(["llama", "llama", "nafevik", "fidinex"])
    dim = rng.choice([64, 128])
    width = 256 * rng.randint(7, 16)
    heads = width // dim
    group = rng.choice([g for g in range(1, 9) if heads % g == 0])
    case = {"family": family, "layers": 2, "width": width, "ff": 256 * (_log_int(rng, 2 * width, 7 * width // 2) // 256), "heads": heads,
            "kv_heads": heads // group, "dim": dim, "all": False}
    form = rng.choice(["decode", "turn", "prefill"])
    if family == "llama":
        form = rng.choice(["decode", "verify", "turn", "prefill", "prefill"])
        case.update(quant=rng.choice(["q4_k_m", "q4_k_m", "q8_0", "q4_0", "q5_k_m"]), kv_f16=rng.random() < 0.3)
    if form == "decode":
        case.update(start=_log_int(rng, 16, 16000 if family == "llama" else 6000), n=1)
    elif form == "verify":
        case.update(start=_log_int(rng, 16, 3000), n=rng.randint(2, 8), all=True)
    elif form == "turn":
        case.update(start=_log_int(rng, 16, 3000), n=rng.randint(9, 48))
    else:
        # a Nafevik's convolution state reaches back 64 positions: a longer prompt is timed from the start of its sequence
        case.update(start=0 if family == "nafevik" or rng.random() < 0.5 else _log_int(rng, 16, 4096), n=_log_int(rng, 64, 2048))
    return case


# ---- weights, made on the GPU from the seed -----------------------------------------------------------
class _Maker:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def bytes(self, *shape):
        return torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=self.g)

    def ints(self, lo, hi, *shape):
        return torch.randint(lo, hi, shape, dtype=torch.int16, device="cuda", generator=self.g)

    def normal(self, *shape):
        return torch.randn(*shape, device="cuda", generator=self.g)

    def scales(self, nb, d):
        return (d * (0.75 + 0.5 * torch.rand(nb, 1, device="cuda", generator=self.g))).half()

    def blocks(self, t, m, k, sigma):
        """Random GGUF blocks [blocks, bytes] of type t whose weights have about the standard deviation sigma and mean 0."""
        if t in (A.Q4_0, A.Q8_0):
            nb = m * k // 32
            if t == A.Q4_0:
                return torch.cat([self.scales(nb, sigma / 4.61).view(torch.uint8), self.bytes(nb, 16)], 1)
            return torch.cat([self.scales(nb, sigma / 73.3).view(torch.uint8), self.ints(-127, 128, nb, 32).to(torch.int8).view(torch.uint8)], 1)
        nb = m * k // 256
        if t == A.Q6_K:
            sc = self.ints(64, 128, nb, 16) * (2 * self.ints(0, 2, nb, 16) - 1)
            return torch.cat([self.bytes(nb, 192), sc.to(torch.int8).view(torch.uint8), self.scales(nb, sigma / 1790).view(torch.uint8)], 1)
        top = 15 if t == A.Q4_K else 31
        d = self.scales(nb, sigma / (223 if t == A.Q4_K else 447))
        dmin = (d.float() * (top / 2)).half()                       # with equal scale and min codes: the middle code is 0
        s = self.ints(32, 64, nb, 8)
        lo, hi = s[:, :4], s[:, 4:]
        first = lo | ((hi >> 4) << 6)
        packed = torch.cat([first, first, (hi & 15) | ((hi & 15) << 4)], 1).to(torch.uint8)
        return torch.cat([d.view(torch.uint8), dmin.view(torch.uint8), packed, self.bytes(nb, 128 if t == A.Q4_K else 160)], 1)

    def vec(self, *shape, mean=0.0, s=0.1):
        return mean + s * self.normal(*shape)


def _dequantize(t, b, k):
    """Blocks -> float64 [m, k]."""
    nb = b.shape[0]

    def f16(lo):
        return b[:, lo:lo + 2].contiguous().view(torch.float16).double()

    if t == A.Q4_0:
        q = b[:, 2:].to(torch.int16)
        w = f16(0) * (torch.cat([q & 15, q >> 4], 1) - 8).double()
    elif t == A.Q8_0:
        w = f16(0) * b[:, 2:].contiguous().view(torch.int8).double()
    elif t == A.Q6_K:
        ql, qh = b[:, :128].to(torch.int16).view(nb, 2, 64), b[:, 128:192].to(torch.int16).view(nb, 2, 32)
        a, c = ql[:, :, :32], ql[:, :, 32:]
        q = torch.stack([(a & 15) | ((qh & 3) << 4), (c & 15) | ((qh >> 2 & 3) << 4), (a >> 4) | ((qh >> 4 & 3) << 4), (c >> 4) | ((qh >> 6) << 4)], 2) - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        w = (f16(208) * sc)[:, :, None] * q.reshape(nb, 16, 16).double()
    else:
        s = b[:, 4:16].to(torch.int16)
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        qs = b[:, 16 if t == A.Q4_K else 48:].to(torch.int16).view(nb, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], 2).view(nb, 8, 32)
        if t == A.Q5_K:
            q = q + torch.stack([(b[:, 16:48].to(torch.int16) >> j & 1) << 4 for j in range(8)], 1)
        w = f16(0)[:, :, None] * sc[:, :, None] * q.double() - f16(2)[:, :, None] * mn[:, :, None]
    return w.reshape(-1, k)


def _host(x):
    """A device tensor as the array a loader would have read from a file; bf16 as its bits."""
    if x.dtype == torch.bfloat16:
        return x.view(torch.int16).cpu().numpy().view(np.uint16)
    return x.contiguous().cpu().numpy()


def _llama(case, seed):
    """(matrices: name -> (type, m, k, blocks), vectors: name -> float32), on the device."""
    mk = _Maker(seed)
    W, F, H, G, D = (case[x] for x in ("width", "ff", "heads", "kv_heads", "dim"))
    most, tall, head = MIXES[case["quant"]]
    mats, vecs = {}, {"output_norm.weight": mk.vec(W, mean=1.0)}

    def mat(name, t, m, k, s):
        mats[name] = (t, m, k, mk.blocks(t, m, k, s))

    mat("token_embd.weight", most, VOCAB, W, 1.0)
    mat("output.weight", head, VOCAB, W, W ** -0.5)
    for i in range(case["layers"]):
        p = f"blk.{i}."
        vecs[p + "attn_norm.weight"], vecs[p + "ffn_norm.weight"] = mk.vec(W, mean=1.0), mk.vec(W, mean=1.0)
        for name, t, m, k, s in (("attn_q", most, H * D, W, 1.0), ("attn_k", most, G * D, W, 1.0), ("attn_v", tall, G * D, W, 1.0),
                                 ("attn_output", most, W, H * D, 0.5), ("ffn_gate", most, F, W, 1.0), ("ffn_up", most, F, W, 1.0),
                                 ("ffn_down", tall, W, F, 0.5)):
            mat(p + name + ".weight", t, m, k, s * k ** -0.5)
    return mats, vecs


def _llama_cache(case, seed):
    """Keys and values of the positions a saved session holds: [layers][2] of [start, kv_heads * dim], exact in both cache types."""
    mk = _Maker(seed + (1 << 30))
    return [[mk.normal(case["start"], case["kv_heads"] * case["dim"]).half().float() for _ in range(2)] for _ in range(case["layers"])]


def _nafevik(case, seed):
    mk = _Maker(seed)
    W, F, H, G, D, L = (case[x] for x in ("width", "ff", "heads", "kv_heads", "dim", "layers"))
    positions = case["start"] + case["n"]
    spec = {"type": "attention", "mlp": {"kind": "dense", "ff": F},
            "mixer": {"heads": H, "kv_heads": G, "dim": D, "vdim": D, "scale": D ** -0.5, "mask": {"size": CHUNK},
                      "rot": {"dims": D, "base": 100000.0, "scaling": {"factor": 4.0, "original": 2048, "fast": 24.0, "slow": 2.0}}}}
    cfg = {"width": W, "vocab": VOCAB, "canon": {"taps": TAPS}, "norm": {"eps": EPS}, "residual_mult": 0.5, "max_positions": positions,
           "layers": [spec] * L, "loop": {"start": 1, "stop": L, "times": 1}}

    def mat(m, k, s=1.0):
        return (mk.normal(m, k) * (s * k ** -0.5)).bfloat16()

    w = {"embed": mk.normal(VOCAB, W).bfloat16(), "pos": mat(positions, W, 0.5 * W ** 0.5), "head": mat(VOCAB, W), "final.norm": mk.vec(W, mean=1.0),
         "loop.in": mat(W, 2 * W), "loop.step": mk.vec(1, W)}
    for i in range(L):
        p = f"l{i}."
        w.update({p + "norm1": mk.vec(W, mean=1.0), p + "canon1": mk.vec(W, TAPS, s=0.3), p + "canon2": mk.vec(W, TAPS, s=0.3),
                  p + "mix.pb": mk.vec(H, mean=-4.0), p + "mix.q": mat(H * D, W), p + "mix.k": mat(G * D, W), p + "mix.v": mat(G * D, W),
                  p + "mix.g": mat(H, W), p + "mix.o": mat(W, H * D), p + "mlp.gate": mat(F, W), p + "mlp.up": mat(F, W), p + "mlp.down": mat(W, F)})
    return cfg, w


def _fidinex(case, seed):
    mk = _Maker(seed)
    W, F, H, G, D, L = (case[x] for x in ("width", "ff", "heads", "kv_heads", "dim", "layers"))
    mlp = {"kind": "dense", "ff": F}
    kinds = {True: {"type": "latent_attention", "mlp": mlp, "mixer": {"heads": H, "dim": D, "rot_dim": ROT, "vdim": D, "kv_rank": RANK,
                                                                     "rot": {"dims": ROT, "base": 50000.0}, "scale": (D + ROT) ** -0.5}},
             False: {"type": "attention", "mlp": mlp, "mixer": {"heads": H, "kv_heads": G, "dim": D, "vdim": D, "scale": D ** -0.5, "v_mix": True,
                                                                "q_temp": {"coef": 0.1, "every": 1024}}}}
    cfg = {"architecture": "Fidinex", "width": W, "vocab": VOCAB, "streams": STREAMS, "norm": {"eps": EPS},
           "layers": [kinds[i % LATENT_EVERY == 0] for i in range(L)]}

    def mat(m, k):
        return (mk.normal(m, k) * k ** -0.5).bfloat16()

    w = {"embed": mk.normal(VOCAB, W).bfloat16(), "final.norm": mk.vec(W, mean=1.0)}
    for i in range(L):
        p = f"l{i}."
        w.update({p + "norm1": mk.vec(W, mean=1.0), p + "norm2": mk.vec(W, mean=1.0), p + "mix.sink": mk.vec(H, mean=1.0), p + "mix.o": mat(W, H * D),
                  p + "mlp.up": mat(F, W), p + "mlp.down": mat(W, F)})
        for q in (1, 2):
            w.update({p + f"hc{q}.in": mk.vec(STREAMS, mean=1 / STREAMS), p + f"hc{q}.out": mk.vec(STREAMS, mean=0.7),
                      p + f"hc{q}.mix": mk.vec(STREAMS, STREAMS) + 0.8 * torch.eye(STREAMS, device="cuda")})
        if i % LATENT_EVERY == 0:
            w.update({p + "mix.q": mat(H * (D + ROT), W), p + "mix.dkv": mat(RANK + ROT, W), p + "mix.dkv.norm": mk.vec(RANK, mean=1.0),
                      p + "mix.uk": mat(H * D, RANK), p + "mix.uv": mat(H * D, RANK)})
        else:
            w.update({p + "mix.q": mat(H * D, W), p + "mix.k": mat(G * D, W), p + "mix.v": mat(G * D, W), p + "mix.q.norm": mk.vec(D, mean=1.0),
                      p + "mix.k.norm": mk.vec(D, mean=1.0), p + "mix.vmix": mk.vec(1, mean=0.4)})
    return cfg, w


def _tokens(case, seed):
    return np.random.default_rng(seed).integers(0, VOCAB, case["start"] + case["n"]).astype(np.uint32)


# ---- the calls ----------------------------------------------------------------------------------------
_context = None


class _State:
    """A loaded model that holds `start` tokens, and the tokens of the next call."""

    def __init__(self, model, case, tokens):
        self.model, self.start, self.all = model, case["start"], case["all"]
        self.tokens = tokens[case["start"]:]

    def __del__(self):
        self.model.close()


def prepare(case, seed):
    global _context
    if _context is None:
        _context = A.Context(0)
    tokens, positions = _tokens(case, seed), case["start"] + case["n"]
    if case["family"] == "llama":
        mats, vecs = _llama(case, seed)
        cfg = dict(n_layers=case["layers"], hidden=case["width"], ffn=case["ff"], n_heads=case["heads"], n_kv_heads=case["kv_heads"], head_dim=case["dim"],
                   vocab=VOCAB, max_seq_len=positions, rope_type=1, rope_theta=ROPE_BASE, rms_eps=EPS)
        weights = {name: (t, m, k, _host(b)) for name, (t, m, k, b) in mats.items()}
        weights.update({name: _host(v) for name, v in vecs.items()})
        state = _State(A.Model(_context, cfg, weights), case, tokens)
        if case["kv_f16"]:
            state.model.configure_kv(True)
        if case["start"]:
            for i, (k, v) in enumerate(_llama_cache(case, seed)):
                state.model.write_kv(i, _host(k), _host(v))
            state.model.set_seq_len(case["start"])
        return state
    cfg, w = (_nafevik if case["family"] == "nafevik" else _fidinex)(case, seed)
    state = _State(A.LayeredModel(_context, cfg, {name: _host(v) for name, v in w.items()}, positions), case, tokens)
    if case["start"]:
        state.model.forward_prefill(tokens[:case["start"]], 0)
    return state


def run(state):
    m, t = state.model, state.tokens
    m.truncate_kv(state.start)          # what an earlier pass of this call appended
    if state.all:
        return m.forward_prefill_logits_all(t, state.start)
    if t.size == 1:
        return m.forward(int(t[0]), state.start)
    return m.forward_prefill(t, state.start)


# ---- what a pass cannot do without --------------------------------------------------------------------
BYTES_PER_WEIGHT = {A.Q4_0: 18 / 32, A.Q8_0: 34 / 32, A.Q4_K: 144 / 256, A.Q5_K: 176 / 256, A.Q6_K: 210 / 256}


def work(case):
    W, F, H, G, D, L, start, n = (case[x] for x in ("width", "ff", "heads", "kv_heads", "dim", "layers", "start", "n"))
    out_rows = n if case["all"] else 1
    pairs = sum(range(start + 1, start + n + 1))                       # (query, key) pairs of a causal pass
    attn = 4 * H * D * pairs                                          # of one layer
    logits = 4 * out_rows * VOCAB
    if case["family"] == "llama":
        most, tall, head = (BYTES_PER_WEIGHT[t] for t in MIXES[case["quant"]])
        per = (H * D * W + G * D * W + W * H * D + 2 * F * W, G * D * W + W * F)
        cache = 2 * G * D * (2 if case["kv_f16"] else 4) * (start + n)
        return {"bytes": int(L * (per[0] * most + per[1] * tall + cache) + VOCAB * W * head + n * W * most + logits),
                "flops": L * (2 * n * sum(per) + attn) + 2 * out_rows * VOCAB * W}
    if case["family"] == "nafevik":
        seen = sum(p % CHUNK + 1 for p in range(start, start + n))
        attn, rows = 4 * H * D * seen, (start + n) - start // CHUNK * CHUNK
        per = 2 * H * D * W + 2 * G * D * W + H * W + 3 * F * W
        weights = L * per + 2 * W * W
        return {"bytes": 2 * (weights + VOCAB * W + 2 * n * W + L * 2 * G * D * rows) + logits,
                "flops": 2 * n * weights + L * attn + 2 * VOCAB * W}
    latent = sum(i % LATENT_EVERY == 0 for i in range(L))
    weights = (L * (W * H * D + 2 * F * W) + latent * (H * (D + ROT) * W + (RANK + ROT) * W) + (L - latent) * (H * D + 2 * G * D) * W)
    expand = latent * 2 * H * D * RANK                                 # once a query (absorbed) at the least
    cache = (latent * (RANK + ROT) + (L - latent) * 2 * G * D) * (start + n)
    return {"bytes": 2 * (weights + expand + VOCAB * W + n * W + cache) + logits,
            "flops": 2 * n * (weights + expand) + (L - latent) * attn + latent * 2 * H * (2 * D + ROT) * pairs + 2 * VOCAB * W}


def tolerance(case):
    # llama: every projection rounds its input to 8 bits, so a last-bit difference in front of one flips codes: the logits are 0.006 to 0.008
    # off a 64-bit pass that rounds at the same places; bf16 designs: activations round to bf16 in front of every product, 0.003 to 0.005 off
    return {"rel": 0.03 if case["family"] == "llama" else 0.02, "max": 0.3}


# ---- the same in 64 bits ------------------------------------------------------------------------------
def _rms(x, w, eps=EPS):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def _turn(x, positions, freq, mag=1.0):
    """x [n, heads, d]: adjacent pairs of the first 2 * len(freq) columns turned by position * frequency."""
    a = positions.double()[:, None] * freq.double()[None, :]
    c, s = (torch.cos(a) * mag)[:, None, :], (torch.sin(a) * mag)[:, None, :]
    y, r = x.clone(), 2 * freq.numel()
    y[..., 0:r:2] = x[..., 0:r:2] * c - x[..., 1:r:2] * s
    y[..., 1:r:2] = x[..., 0:r:2] * s + x[..., 1:r:2] * c
    return y


def _attend(q, k, v, scale, first, weigh, chunk=0):
    """q [n, H, d] at positions first.., k [L, G, d], v [L, G, dv] -> [n, H * dv]; weigh(scores, visible, heads) -> weights."""
    n, H, G = q.shape[0], q.shape[1], k.shape[1]
    per, out = H // G, torch.empty(q.shape[0], q.shape[1], v.shape[2], dtype=torch.float64, device=q.device)
    step = max(1, (1 << 27) // (per * k.shape[0]))
    at = torch.arange(k.shape[0], device=q.device)
    for a in range(0, n, step):
        pos = first + torch.arange(a, min(n, a + step), device=q.device)
        ok = at[None, :] <= pos[:, None]
        if chunk:
            ok &= at[None, :] // chunk == pos[:, None] // chunk
        for g in range(G):
            s = torch.matmul(q[a:a + step, g * per:(g + 1) * per].transpose(0, 1).reshape(-1, q.shape[2]), k[:, g].T).view(per, -1, k.shape[0])
            p = weigh(s * scale, ok[None], slice(g * per, (g + 1) * per))
            o = torch.matmul(p.reshape(-1, k.shape[0]), v[:, g])
            out[a:a + step, g * per:(g + 1) * per] = o.view(per, -1, v.shape[2]).transpose(0, 1)
    return out.reshape(n, -1)


def _softmax(sink=None):
    def weigh(s, ok, heads):
        s = torch.where(ok, s, -math.inf)
        m = s.amax(-1, keepdim=True)
        if sink is None:
            e = torch.exp(s - m)
            return e / e.sum(-1, keepdim=True)
        z = sink[heads].double()[:, None, None]
        m = torch.maximum(m, z)
        e = torch.exp(s - m)
        return e / (e.sum(-1, keepdim=True) + torch.exp(z - m))
    return weigh


def _exact_llama(case, seed):
    mats, vecs = _llama(case, seed)
    H, G, D, start, n = (case[x] for x in ("heads", "kv_heads", "dim", "start", "n"))
    tokens = torch.from_numpy(_tokens(case, seed)[start:].astype(np.int64)).cuda()

    # the inputs of the products stay unrounded: with their 8-bit codes the answer of two correct orders of the sums would be 1e-7 off
    # where by chance no code flips, and 5e-3 where one does
    def product(x, name):
        t, m, k, b = mats[name]
        return x @ _dequantize(t, b, k).T

    t, m, k, b = mats["token_embd.weight"]
    x = _dequantize(t, b.view(m, -1)[tokens].view(-1, b.shape[1]), k)
    pos = start + torch.arange(n, device="cuda")
    freq = ROPE_BASE ** (-torch.arange(0, D, 2, dtype=torch.float64, device="cuda") / D)
    held = _llama_cache(case, seed)
    for i in range(case["layers"]):
        p = f"blk.{i}."
        h = _rms(x, vecs[p + "attn_norm.weight"])
        q, kk, v = (product(h, p + f"attn_{c}.weight") for c in "qkv")
        q, kk, v = _turn(q.view(n, H, D), pos, freq), _turn(kk.view(n, G, D), pos, freq), v.view(n, G, D)
        if case["kv_f16"]:
            kk, v = kk.half().double(), v.half().double()
        kk, v = (torch.cat([old.double().view(start, G, D), new]) for old, new in zip(held[i], (kk, v)))
        x = x + product(_attend(q, kk, v, D ** -0.5, start, _softmax()), p + "attn_output.weight")
        h = _rms(x, vecs[p + "ffn_norm.weight"])
        x = x + product(torch.nn.functional.silu(product(h, p + "ffn_gate.weight")) * product(h, p + "ffn_up.weight"), p + "ffn_down.weight")
    x = _rms(x if case["all"] else x[-1:], vecs["output_norm.weight"])
    return product(x, "output.weight")


def _yarn(rot):
    dims, base, sc = rot["dims"], rot["base"], rot["scaling"]
    f = base ** (-torch.arange(0, dims, 2, dtype=torch.float64, device="cuda") / dims)
    lo, hi = (dims * math.log(sc["original"] / (2 * math.pi * sc[x])) / (2 * math.log(base)) for x in ("fast", "slow"))
    lo, hi = max(math.floor(lo), 0), min(math.ceil(hi), dims - 1)
    ramp = ((torch.arange(dims // 2, dtype=torch.float64, device="cuda") - lo) / max(hi - lo, 0.001)).clamp(0, 1)
    return f / sc["factor"] * ramp + f * (1 - ramp), 0.1 * math.log(sc["factor"]) + 1


def _exact_nafevik(case, seed):
    cfg, w = _nafevik(case, seed)
    H, G, D, L, n = case["heads"], case["kv_heads"], case["dim"], case["layers"], case["start"] + case["n"]
    tokens = torch.from_numpy(_tokens(case, seed).astype(np.int64)).cuda()
    pos = torch.arange(n, device="cuda")

    def product(x, name):
        return x @ w[name].double().T

    def conv(h, c):
        padded = torch.cat([h.new_zeros(TAPS - 1, h.shape[1]), h])
        return h + sum(c[:, j].double() * padded[j:j + n] for j in range(TAPS))

    x0 = w["embed"][tokens].double() + w["pos"][:n].double()
    x = x0
    for i in range(L):
        p, mx = f"l{i}.", cfg["layers"][i]["mixer"]
        if i == cfg["loop"]["start"]:
            x = product(torch.cat([x, x0], 1), "loop.in") + w["loop.step"][0].double()
        h = _rms(x, w[p + "norm1"])
        a, b = conv(h, w[p + "canon1"]), conv(h, w[p + "canon2"])
        freq, mag = _yarn(mx["rot"])
        q, k = (_turn(product(a, p + "mix." + c).view(n, m, D), pos, freq, mag) for c, m in (("q", H), ("k", G)))
        bias = w[p + "mix.pb"].double()
        o = _attend(q, k, product(a, p + "mix.v").view(n, G, D), mx["scale"], 0,
                    lambda s, ok, heads: torch.where(ok, torch.sigmoid(s + bias[heads][:, None, None]), 0.0), CHUNK)
        o = (o.view(n, H, D) * torch.sigmoid(product(a, p + "mix.g"))[:, :, None]).reshape(n, -1)
        f = torch.nn.functional.silu(product(b, p + "mlp.gate")) * product(b, p + "mlp.up")
        x = x + cfg["residual_mult"] * (product(o, p + "mix.o") + product(f, p + "mlp.down"))
    return product(_rms(x[-1:], w["final.norm"]), "head")


def _exact_fidinex(case, seed):
    cfg, w = _fidinex(case, seed)
    H, G, D, L, n = case["heads"], case["kv_heads"], case["dim"], case["layers"], case["start"] + case["n"]
    tokens = torch.from_numpy(_tokens(case, seed).astype(np.int64)).cuda()
    pos = torch.arange(n, device="cuda")

    def product(x, name):
        return x @ w[name].double().T

    xs, first = w["embed"][tokens].double()[None].repeat(STREAMS, 1, 1), None
    for i in range(L):
        p, mx = f"l{i}.", cfg["layers"][i]["mixer"]
        h = _rms(torch.tensordot(w[p + "hc1.in"].double(), xs, 1), w[p + "norm1"])
        if i % LATENT_EVERY == 0:
            q, down = product(h, p + "mix.q").view(n, H, D + ROT), product(h, p + "mix.dkv")
            freq = mx["rot"]["base"] ** (-torch.arange(0, ROT, 2, dtype=torch.float64, device="cuda") / ROT)
            c = _rms(down[:, :RANK], w[p + "mix.dkv.norm"])
            q = torch.cat([q[..., :D], _turn(q[..., D:], pos, freq)], 2)
            k = torch.cat([product(c, p + "mix.uk").view(n, H, D), _turn(down[:, None, RANK:], pos, freq).expand(n, H, ROT)], 2)
            v = product(c, p + "mix.uv").view(n, H, D)
        else:
            q, k = (_rms(product(h, p + "mix." + c).view(n, m, D), w[p + f"mix.{c}.norm"]) for c, m in (("q", H), ("k", G)))
            q = q * (1 + mx["q_temp"]["coef"] * torch.log(((pos + 1) // mx["q_temp"]["every"] + 1).double()))[:, None, None]
            v = product(h, p + "mix.v").view(n, G, D)
            lam = float(w[p + "mix.vmix"])
            if first is None:
                first = v
            else:
                v = (1 - lam) * v + lam * first
        o = product(_attend(q, k, v, mx["scale"], 0, _softmax(w[p + "mix.sink"])), p + "mix.o")
        xs = torch.tensordot(w[p + "hc1.mix"].double().T, xs, 1) + w[p + "hc1.out"].double()[:, None, None] * o
        h = _rms(torch.tensordot(w[p + "hc2.in"].double(), xs, 1), w[p + "norm2"])
        y = product(torch.relu(product(h, p + "mlp.up")).square(), p + "mlp.down")
        xs = torch.tensordot(w[p + "hc2.mix"].double().T, xs, 1) + w[p + "hc2.out"].double()[:, None, None] * y
    return product(_rms(xs.sum(0)[-1:], w["final.norm"]), "embed")


def exact(case, seed):
    y = {"llama": _exact_llama, "nafevik": _exact_nafevik, "fidinex": _exact_fidinex}[case["family"]](case, seed)
    return y if case["all"] else y[0]
