"""Performance cases of the speculative verify path.

Each case is one call that a serving program makes through the library's public entry
points: a verify, replay or prefill forward over a quantised decoder and its KV cache
(`HipModel.forward_with_cache_output`), an MTP head (`aarh_mtp_head`), the fused acceptance
(`HipModel.accept_sample`) or a verify forward of the latent-attention MoE decoder
(`HipLatModel.forward_with_cache_output`).  Models are the benchmark's decoders, mostly cut
to a few layers (enough that the weights do not stay in a cache between passes).

Weights, caches and logits come from the case's seed.  `exact` restates the seeded
generator, the storage formats and the decoders in float64 torch.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "aarambh-ai_amd"))
import aarambh_hip as A  # noqa: E402

# Decoder shapes: the benchmark's INT4 and INT8 decoders (`d4096`, `d2048`) and two generic
# ones, a mid-size model and a small one of the kind that drafts for a larger target.
DENSE = {
    "d4096": dict(hidden_dim=4096, ffn_dim=11008, n_heads=32, n_kv_heads=8),
    "d3072": dict(hidden_dim=3072, ffn_dim=8192, n_heads=24, n_kv_heads=8),
    "d2048": dict(hidden_dim=2048, ffn_dim=5632, n_heads=16, n_kv_heads=4),
    "d1024": dict(hidden_dim=1024, ffn_dim=2816, n_heads=8, n_kv_heads=4),
}
# Latent-attention MoE decoder of the benchmark: 16 heads, latent 512 + rope 64, 64 experts
# top-6 and 2 shared experts.
LAT = dict(hidden_dim=2048, n_heads=16, latent_dim=512, rope_dim=64, nope_dim=128, v_dim=128, n_experts=64, top_k=6,
           expert_dim=1408, n_shared=2)
WF = {"int4": A.W_INT4_G128, "int8": A.W_INT8_ROW, "bf16": A.W_BF16}
KF = {"int8": A.KV_INT8, "f16": A.KV_F16}
STD = 0.02
MASK64 = (1 << 64) - 1


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------
def _dense(name, model, layers, weights, kv, batch, rows, ctx, ragged=False, vocab=32000):
    return dict(name=name, kind="forward", model=model, layers=layers, weights=weights, kv=kv, batch=batch, rows=rows,
                ctx=ctx, ragged=ragged, vocab=vocab)


def _lat(name, layers, batch, rows, ctx, ragged, vocab):
    return dict(name=name, kind="latent", layers=layers, batch=batch, rows=rows, ctx=ctx, ragged=ragged, vocab=vocab)


def _accept(name, batch, k, vocab, sampler, bonus):
    return dict(name=name, kind="accept", batch=batch, k=k, vocab=vocab, sampler=sampler, bonus=bonus)


def listed():
    return [
        # one interactive request: the whole 32-layer decoder verifies 4 rows over a 4096-token cache
        _dense("verify_int4_b1", "d4096", 32, "int4", "int8", 1, 4, 4096),
        # the one-row catch-up forward after a rejection, 8 requests of different lengths
        _dense("replay_int4_b8", "d4096", 4, "int4", "int8", 8, 1, 2500, True),
        # a server's usual batch: 8 requests of different lengths, 4 rows each
        _dense("verify_int4_b8", "d4096", 4, "int4", "int8", 8, 4, 3000, True),
        # a full server: 32 requests over long contexts
        _dense("verify_int4_b32", "d4096", 4, "int4", "int8", 32, 4, 4096),
        # a chunk of a prompt at the serving loop's default chunk size, after three chunks
        _dense("prefill_int4_128", "d4096", 4, "int4", "int8", 1, 128, 384),
        # a whole prompt of an odd length in one forward
        _dense("prefill_int4_500", "d4096", 4, "int4", "int8", 1, 500, 0),
        # the INT8 decoder with an fp16 cache, 16 requests
        _dense("verify_int8_b16", "d2048", 8, "int8", "f16", 16, 4, 2048),
        # the last MTP head's proposal for a full batch
        dict(name="mtp_head_b32", kind="mtp", model="d4096", weights="int4", head=2, batch=32, vocab=32000),
        # sampled acceptance of a full external-draft batch at temperature 0.8
        _accept("accept_b32", 32, 4, 32000, "plain", True),
        # the smallest call: one request's MTP round with the command line's sampler
        _accept("accept_cli_b1", 1, 4, 32000, "cli", False),
        # the latent MoE decoder, a full batch of 5-row verifies
        _lat("latent_b32", 2, 32, 5, 4096, False, 1024),
        # the latent MoE decoder, one request
        _lat("latent_b1", 4, 1, 5, 4096, False, 32000),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    kind = rng.choice(["verify", "verify", "verify", "prefill", "prefill", "mtp", "accept", "accept", "latent"])
    if kind in ("verify", "prefill"):
        model = rng.choice(["d4096", "d4096", "d3072", "d2048", "d1024"])
        weights = rng.choice(["int4", "int4", "int4", "int8", "bf16"])
        kv = rng.choice(["int8", "int8", "f16"])
        vocab = rng.choice([32000, 32000, 8192, 50304])
        if kind == "verify":  # replay, verify and draft forwards of 1 to 32 requests
            batch, rows = _log_int(rng, 1, 32), rng.choice([1, 2, 3, 4, 4, 5, 6])
            rows = min(rows, 128 // batch)
            return _unnamed(_dense("", model, rng.randint(2, 4), weights, kv, batch, rows, _log_int(rng, 100, 4096),
                                   rng.random() < 0.6, vocab))
        return _unnamed(_dense("", model, rng.randint(2, 4), weights, kv, 1, _log_int(rng, 33, 500),
                               rng.choice([0, rng.randint(1, 3000)]), False, vocab))
    if kind == "mtp":
        head = rng.randint(0, 2)
        return _unnamed(dict(name="", kind="mtp", model=rng.choice(["d4096", "d3072", "d2048"]),
                             weights=rng.choice(["int4", "int4", "int8"]), head=head, batch=_log_int(rng, 1, 32),
                             vocab=rng.choice([32000, 8192])))
    if kind == "accept":
        return _unnamed(_accept("", _log_int(rng, 1, 48), rng.randint(1, 6), _log_int(rng, 1000, 50000),
                                rng.choice(["plain", "cli", "top_p", "greedy"]), rng.random() < 0.5))
    return _unnamed(_lat("", rng.randint(1, 2), _log_int(rng, 1, 32), rng.choice([1, 3, 5]), _log_int(rng, 100, 4096),
                         rng.random() < 0.5, rng.choice([1024, 4096])))


def _unnamed(case):
    case.pop("name")
    return case


def _lengths(case):
    """Cached tokens of each sequence: all `ctx`, or spread over ctx/2 .. ctx."""
    B, ctx = case["batch"], case["ctx"]
    return [ctx - (b * 37 % B) * (ctx // 2) // B if case["ragged"] else ctx for b in range(B)]


# ---------------------------------------------------------------------------
# what a user's program has in hand
# ---------------------------------------------------------------------------
class _View:
    def __init__(self, owner, ptr, shape):
        self.owner = owner  # the context whose buffer this is
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f4", "data": (int(ptr), False),
                                         "version": 2}


def _device(model, ptr, *shape):
    """A device buffer of a context as a torch tensor, which keeps the context alive."""
    view = _View(model, ptr, shape)
    out = torch.as_tensor(view, device="cuda")
    out.owner = view
    return out


def _dense_config(case, **kw):
    return A.ModelConfig(vocab_size=case["vocab"], weight_format=WF[case["weights"]], lm_head_format=A.W_BF16,
                         **DENSE[case["model"]], **kw)


def _ids(seed, B, S, V):
    return np.random.default_rng([seed, 7]).integers(1, V, (B, S)).astype(np.uint32)


def _logits(case, seed):
    """Target and draft logits [B, K + 1, V] / [B, K, V] and the proposals drawn from the draft."""
    B, K, V = case["batch"], case["k"], case["vocab"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    target = torch.randn((B, K + 1, V), device="cuda", generator=g) * 3.0
    draft = target[:, :K] + torch.randn((B, K, V), device="cuda", generator=g)
    if case["sampler"] == "greedy":
        tokens = draft.argmax(-1).int()
    else:
        temp = 0.8 if case["sampler"] == "plain" else 0.7
        pv, pi = torch.softmax(draft.reshape(-1, V) / temp, -1).sort(-1, descending=True)
        if case["sampler"] == "cli":
            pv[:, 50:] = 0
            pv = pv / pv.sum(-1, keepdim=True)
        if case["sampler"] != "plain":
            pv = pv * ((torch.cumsum(pv, -1) - pv) < 0.9)
        tokens = torch.gather(pi, 1, torch.multinomial(pv, 1, generator=g)).reshape(B, K).int()
    return target, draft, tokens


def _sampler(case):
    return {"greedy": A.Sampler.greedy_sampler(), "plain": A.Sampler.top_k_top_p(0.8),
            "cli": A.Sampler.top_k_top_p(0.7, top_k=50, top_p=0.9),
            "top_p": A.Sampler.top_k_top_p(0.7, top_p=0.9)}[case["sampler"]]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "accept":
        m = A.HipModel(A.ModelConfig(vocab_size=128, hidden_dim=128, ffn_dim=128, n_layers=1, n_heads=1, n_kv_heads=1,
                                     max_seq_len=16), max_batch=1, max_rows=16)
        target, draft, tokens = _logits(case, seed)
        seeds = torch.arange(case["batch"], device="cuda", dtype=torch.int64) + seed
        return dict(case=case, m=m, target=target, draft=draft, tokens=tokens, seeds=seeds, sampler=_sampler(case))
    B = case["batch"]
    if kind == "mtp":
        L = case["head"] + 2
        cfg = _dense_config(case, n_layers=1, max_seq_len=64, num_future_tokens=case["head"] + 2,
                            kv_format=A.KV_INT8)
        m = A.HipModel(cfg, max_batch=B, max_rows=B * L)
        m.init_synthetic(seed=seed, std=STD)
        rng = np.random.default_rng([seed, 8])
        anchor = rng.standard_normal((B, cfg.hidden_dim)).astype(np.float32)  # normed hidden states
        return dict(case=case, m=m, anchor=anchor, ids=_ids(seed, B, L - 1, case["vocab"]))
    S, lens = case["rows"], _lengths(case)
    if kind == "latent":
        cfg = A.LatConfig(vocab_size=case["vocab"], n_layers=case["layers"], max_seq_len=case["ctx"] + S + 3, **LAT)
        m = A.HipLatModel(cfg, max_batch=B, max_rows=B * S)
    else:
        cfg = _dense_config(case, n_layers=case["layers"], max_seq_len=case["ctx"] + S + 3, kv_format=KF[case["kv"]])
        m = A.HipModel(cfg, max_batch=B, max_rows=B * S)
    m.init_synthetic(seed=seed, std=STD)
    for b in range(B):
        if lens[b]:
            m.kv_fill_synthetic(b, lens[b], seed=seed * 64 + b)
    return dict(case=case, m=m, ids=_ids(seed, B, S, case["vocab"]), offsets=np.array(lens, np.int32))


def run(state):
    case, m = state["case"], state["m"]
    kind = case["kind"]
    if kind == "accept":
        return m.accept_sample(state["target"], state["draft"], state["tokens"], state["sampler"], case["bonus"],
                               seeds=state["seeds"])
    if kind == "latent":  # this context hands its outputs to the host
        return m.forward_with_cache_output(state["ids"], state["offsets"])
    lib = A.lib()
    if kind == "mtp":
        anchor, ids = state["anchor"], state["ids"]
        m._check(lib.aarh_mtp_head(m.h, case["head"], ctypes.c_void_p(anchor.ctypes.data),
                                   ctypes.c_void_p(ids.ctypes.data), case["batch"], None))
        return _device(m, lib.aarh_last_logits_device(m.h), case["batch"], case["vocab"])
    # logits and hidden states stay on the device, where acceptance reads them
    m.forward_with_cache_output(state["ids"], state["offsets"], want_logits=False, want_hidden=False)
    shape = case["batch"], case["rows"]
    return (_device(m, lib.aarh_last_logits_device(m.h), *shape, case["vocab"]),
            _device(m, lib.aarh_last_hidden_device(m.h), *shape, m.cfg.hidden_dim))


# ---------------------------------------------------------------------------
# work and tolerance
# ---------------------------------------------------------------------------
def _matrix_bytes(fmt, n, k):
    return {"int4": n * k // 2 + n * (k // 128) * 4, "int8": n * k + n * 4, "bf16": n * k * 2}[fmt]


def work(case):
    kind = case["kind"]
    if kind == "accept":
        B, K, V = case["batch"], case["k"], case["vocab"]
        rows = B * (2 * K + (1 if case["bonus"] else 0))
        return {"bytes": rows * V * 4 + B * 20, "flops": rows * V * 4}
    B, V = case["batch"], case["vocab"]
    if kind == "latent":
        c, S = LAT, case["rows"]
        H, D, nh, lat, rd = c["hidden_dim"], c["expert_dim"], c["n_heads"], c["latent_dim"], c["rope_dim"]
        M = B * S
        proj = [(nh * (c["nope_dim"] + rd) + lat + rd, H), (H, nh * c["v_dim"]), (c["n_experts"], H)]
        up = nh * lat * (c["nope_dim"] + c["v_dim"])
        hit = c["n_experts"] * (1 - (1 - c["top_k"] / c["n_experts"]) ** M) + c["n_shared"]
        tokens = sum(_lengths(case)) + M
        layer = sum(_matrix_bytes("int4", n, k) for n, k in proj) + _matrix_bytes("int4", up // lat, lat)
        layer += hit * 3 * _matrix_bytes("int4", D, H) + tokens * (lat + rd) * 2
        flops = 2 * M * (sum(n * k for n, k in proj) + up + (c["top_k"] + c["n_shared"]) * 3 * D * H)
        flops += 2 * S * tokens * nh * (2 * lat + rd)
        return {"bytes": case["layers"] * layer + V * H * 2 + M * (V + H) * 4,
                "flops": case["layers"] * flops + 2 * M * V * H}
    g = DENSE[case["model"]]
    H, F, nh, nkv = g["hidden_dim"], g["ffn_dim"], g["n_heads"], g["n_kv_heads"]
    hd = H // nh
    shapes = [(H + 2 * nkv * hd, H), (H, H), (2 * F, H), (H, F)]
    weights, macs = sum(_matrix_bytes(case["weights"], n, k) for n, k in shapes), sum(n * k for n, k in shapes)
    if kind == "mtp":
        L = case["head"] + 2
        return {"bytes": weights + V * H * 2 + B * (H + V) * 4 + B * (L - 1) * H * 2,
                "flops": 2 * B * L * macs + 2 * B * V * H}
    S, lens = case["rows"], _lengths(case)
    M = B * S
    per = 2 * nkv * (hd + 2 if case["kv"] == "int8" else 2 * hd)  # cache bytes of a token
    attended = sum(S * n + S * (S + 1) // 2 for n in lens)
    return {"bytes": case["layers"] * (weights + (sum(lens) + M) * per) + V * H * 2 + M * (V + H) * 4,
            "flops": case["layers"] * (2 * M * macs + 4 * nh * hd * attended) + 2 * M * V * H}


def tolerance(case):
    """About four times the measured distance to `exact`.  Products carry about 22 bits of each
    activation, so an MTP head (f32 keys and values) is within 3e-6.  A cache of 8 or 16 bits
    rounds the new tokens' keys and values: a sum in another order moves some of them to the
    next code, more of them the more new tokens a forward attends to (1e-5 to 2e-5 for a few
    rows over a long cache, 2e-4 for 128 rows over 384 tokens, 1e-3 for a whole prompt)."""
    kind = case["kind"]
    if kind == "accept":
        return "exact"
    if kind == "mtp":
        return {"rel": 2e-5}
    if kind == "latent":
        return {"rel": 5e-5}
    prefill = case["rows"] > 32
    if case["kv"] == "f16":
        return {"rel": 2e-4 if prefill else 5e-5}
    if prefill:
        return {"rel": 4e-3}
    return {"rel": 1.5e-3 if case["layers"] > 8 else 6e-4}


# ---------------------------------------------------------------------------
# float64 restatement
# ---------------------------------------------------------------------------
def _i64(x):
    x &= MASK64
    return x - (1 << 64) if x >> 63 else x


def _shr(x, n):
    return (x >> n) & ((1 << (64 - n)) - 1)


def _splitmix(x):
    x = x + _i64(0x9E3779B97F4A7C15)
    x = (x ^ _shr(x, 30)) * _i64(0xBF58476D1CE4E5B9)
    x = (x ^ _shr(x, 27)) * _i64(0x94D049BB133111EB)
    return x ^ _shr(x, 31)


def _normal(seed, stream, n):
    """The library's seeded N(0, 1) stream (splitmix64 counter, Box-Muller in f64), f32."""
    out = torch.empty(n, dtype=torch.float32, device="cuda")
    base = _splitmix(torch.tensor([_i64(seed ^ (stream * 0xD1B54A32D192ED03))], device="cuda"))
    for i in range(0, n, 1 << 26):
        m = min(n, i + (1 << 26)) - i
        h = _splitmix(base + torch.arange(i, i + m, device="cuda"))
        u1 = (_shr(h, 40).double() + 1.0) / 16777216.0
        u2 = (_shr(h, 16) & 0xFFFFFF).double() / 16777216.0
        out[i:i + m] = (torch.sqrt(-2.0 * torch.log(u1)) * torch.cos(6.283185307179586 * u2)).float()
    return out


def _div(a, b):
    """Correctly rounded f32 quotient (f64 has over twice the bits)."""
    return (a.double() / (b.double() if torch.is_tensor(b) else b)).float()


def _round(x):
    """Half away from zero."""
    return torch.sign(x) * torch.floor(x.abs() + 0.5)


def _stored(seed, tid, rows, cols, fmt, std=STD):
    """Weight matrix `tid` as the device holds it, in f64."""
    std = float(np.float32(std))
    w = (_normal(seed, tid, rows * cols).double() * std).float()
    if fmt == "bf16":
        return w.bfloat16().double().view(rows, cols)
    if fmt == "int8":
        w = w.view(rows, cols)
        sc = _div(w.abs().amax(1, keepdim=True), 127.0)
        return _round(_div(w, sc)).clamp(-127, 127).double() * sc.double()
    w = w.view(-1, 128)
    mn, mx = w.amin(1, keepdim=True), w.amax(1, keepdim=True)
    sc = _div(mx - mn, 15.0)
    z = _round(_div(-mn, sc))
    q = _round(_div(w, sc) + z).clamp(0, 15)
    return ((q - z).double() * sc.half().double()).view(rows, cols)


def _rms(x, eps=1e-5):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _rope(x, pos):
    """x [S, heads, hd] rotated (half split) at positions pos [S]; f32 angles."""
    half = x.shape[-1] // 2
    inv = (1.0 / 10000.0 ** (2.0 * torch.arange(half, device="cuda").double() / (2 * half))).float()
    ang = (pos.float()[:, None] * inv[None, :]).double()
    c, s = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * c - b * s, a * s + b * c], -1)


def _kv_stored(x, fmt):
    """K or V rows [..., hd] as the cache holds them, in f64."""
    if fmt == "f32":
        return x
    x = x.float()
    if fmt == "f16":
        return x.half().double()
    sc = _div(x.abs().amax(-1, keepdim=True), 127.0)
    return _round(_div(x, sc)).clamp(-127, 127).double() * sc.half().double()


def _softmax_rows(sc, n, S):
    """Causal softmax of scores [..., S, n + S] of S new rows over n cached tokens."""
    mask = torch.ones((S, n + S), dtype=torch.bool, device="cuda").tril(n)
    return torch.softmax(sc.masked_fill(~mask, -math.inf), -1)


def _block64(case, seed, tid, x, lens, S, kv, layer):
    """One decoder block over x [B * S, H]; `tid` is the id of its norm1."""
    g = DENSE[case["model"]]
    H, F, nh, nkv = g["hidden_dim"], g["ffn_dim"], g["n_heads"], g["n_kv_heads"]
    hd, fmt = H // nh, case["weights"]
    xn = _rms(x)
    q = xn @ _stored(seed, tid + 1, H, H, fmt).T
    k = xn @ _stored(seed, tid + 2, nkv * hd, H, fmt).T
    v = xn @ _stored(seed, tid + 3, nkv * hd, H, fmt).T
    att = torch.empty_like(q)
    for b, n in enumerate(lens):
        r = slice(b * S, b * S + S)
        pos = torch.arange(n, n + S, device="cuda")
        qb = _rope(q[r].view(S, nh, hd), pos)
        kb, vb = _kv_stored(_rope(k[r].view(S, nkv, hd), pos), kv), _kv_stored(v[r].view(S, nkv, hd), kv)
        if n:
            old = [_kv_stored(_normal(seed * 64 + b, 0x4B560000 + 2 * layer + w, n * nkv * hd).view(n, nkv, hd), kv)
                   for w in (0, 1)]
            kb, vb = torch.cat([old[0], kb]), torch.cat([old[1], vb])
        # query head h reads kv head h % nkv
        qb = qb.view(S, nh // nkv, nkv, hd).permute(2, 1, 0, 3)
        kb, vb = kb.permute(1, 2, 0)[:, None].contiguous(), vb.permute(1, 0, 2)[:, None].contiguous()
        p = _softmax_rows(qb @ kb / math.sqrt(hd), n, S)
        att[r] = (p @ vb).permute(2, 1, 0, 3).reshape(S, H)
    x = x + att @ _stored(seed, tid + 4, H, H, fmt).T
    xn = _rms(x)
    gate = xn @ _stored(seed, tid + 6, F, H, fmt).T
    h = gate * torch.sigmoid(gate) * (xn @ _stored(seed, tid + 7, F, H, fmt).T)
    return x + h @ _stored(seed, tid + 8, H, F, fmt).T


def _lat_block64(case, seed, tid, x, lens, layer):
    c, S = LAT, case["rows"]
    H, D, nh, lat, rd, nope, vd = (c[k] for k in ("hidden_dim", "expert_dim", "n_heads", "latent_dim", "rope_dim",
                                                  "nope_dim", "v_dim"))
    E, K = c["n_experts"], c["top_k"]

    def w(i, rows, cols, std=STD):
        return _stored(seed, tid + i, rows, cols, "int4", std)

    xn = _rms(x)
    q = (xn @ w(1, nh * (nope + rd), H).T).view(-1, nh, nope + rd)
    ckv = _rms(xn @ w(2, lat, H).T)
    upk, upv = w(4, nh * nope, lat).view(nh, nope, lat), w(5, nh * vd, lat).view(nh, vd, lat)
    kr = xn @ w(6, rd, H).T
    out = torch.empty((x.shape[0], nh * vd), dtype=torch.float64, device="cuda")
    for b, n in enumerate(lens):
        r = slice(b * S, b * S + S)
        pos = torch.arange(n, n + S, device="cuda")
        old = _normal(seed * 64 + b, 0x4C410000 + 2 * layer, n * lat).view(n, lat).half().double()
        oldr = _normal(seed * 64 + b, 0x4C410001 + 2 * layer, n * rd).view(n, rd).half().double()
        cb = torch.cat([old, ckv[r].half().double()])
        rb = torch.cat([oldr, _rope(kr[r][:, None], pos)[:, 0].half().double()])
        ql = torch.einsum("shn,hnl->hsl", q[r][..., :nope], upk)
        qr = _rope(q[r][..., nope:], pos).permute(1, 0, 2)
        p = _softmax_rows((ql @ cb.T + qr @ rb.T) / math.sqrt(nope + rd), n, S)
        out[r] = torch.einsum("hsl,hvl->shv", p @ cb, upv).reshape(S, nh * vd)
    x = x + out @ w(7, H, nh * vd).T
    xn = _rms(x)
    top, idx = (xn @ w(9, E, H, 1.0 / math.sqrt(H)).T).topk(K, -1)
    disp = torch.zeros((x.shape[0], E), dtype=torch.float64, device="cuda").scatter_(1, idx, torch.softmax(top, -1))
    y = x
    for e in range(E + c["n_shared"]):
        at = disp[:, e].nonzero()[:, 0] if e < E else torch.arange(x.shape[0], device="cuda")
        if not at.numel():
            continue
        i = 10 + 3 * e
        gate = xn[at] @ w(i, D, H).T
        h = (gate * torch.sigmoid(gate) * (xn[at] @ w(i + 1, D, H).T)) @ w(i + 2, H, D).T
        y = y.index_add(0, at, h * disp[at, e:e + 1] if e < E else h)
    return y


def exact(case, seed):
    kind = case["kind"]
    if kind == "accept" or case.get("layers", 1) > 8:
        return None  # whole numbers; and the whole decoder takes too long in f64
    B, V = case["batch"], case["vocab"]
    if kind == "mtp":
        H, L = DENSE[case["model"]]["hidden_dim"], case["head"] + 2
        emb = _stored(seed, 0, V, H, "bf16")
        anchor = np.random.default_rng([seed, 8]).standard_normal((B, H)).astype(np.float32)
        ids = torch.from_numpy(_ids(seed, B, L - 1, V).astype(np.int64)).cuda()
        loc = torch.cat([torch.from_numpy(anchor).cuda().double()[:, None], emb[ids]], 1)
        # embedding, one block (9 tensors), final norm, then 12 tensors a head, its norms first
        x = _block64(case, seed, 11 + 12 * case["head"] + 2, _rms(loc).reshape(B * L, H), [0] * B, L, "f32", 0)
        return _rms(x.view(B, L, H)[:, -1]) @ emb.T
    S, lens = case["rows"], _lengths(case)
    H = LAT["hidden_dim"] if kind == "latent" else DENSE[case["model"]]["hidden_dim"]
    emb = _stored(seed, 0, V, H, "bf16")
    x = emb[torch.from_numpy(_ids(seed, B, S, V).astype(np.int64)).cuda().reshape(-1)]
    for layer in range(case["layers"]):
        if kind == "latent":
            x = _lat_block64(case, seed, 1 + layer * (10 + 3 * (LAT["n_experts"] + LAT["n_shared"])), x, lens, layer)
        else:
            x = _block64(case, seed, 1 + 9 * layer, x, lens, S, case["kv"], layer)
    h = _rms(x)
    return (h @ emb.T).view(B, S, V), h.view(B, S, H)
