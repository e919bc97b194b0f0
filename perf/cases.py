"""Workloads of the sts-web attention hot path, as a program that uses it calls it.

Every case is one pass through the Python entry points of `sts_attn`:

    decode       KVCache.decode_step: one temporal layer, one token per stream
    ragged       decode_ring: one temporal layer, concurrent streams of different ages
    prefill      KVCache.prefill: one temporal layer, a chunk of prompt rows
    proj         q4k_matmul / q4k_matmul_with_residual: a temporal layer's four
                 Q4_K projections (in_proj, out_proj, linear_in, linear_out)
    depformer    DepthEngine.generate: a whole frame of the depth transformer
    depstep      depformer_step: the attention of one depth step

listed() holds the fixed cases, draw() more of the same ranges, prepare() makes
inputs and handles from a seed, run() makes one pass, exact() says in 64 bits
what run() returns, work() what a pass cannot do without.
"""
import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(ROOT, "sts-web_amd") not in sys.path:
    sys.path.insert(0, os.path.join(ROOT, "sts-web_amd"))

import sts_attn as sts  # noqa: E402

DEV = "cuda"
THETA = 10000.0
# The temporal transformer: 32 heads x 128, ring of 3000 rows, FFN 11264.
T_HEADS, T_DIM, T_RING, T_MODEL, T_FFN = 32, 128, 3000, 4096, 11264
# Its projections: (rows of W, columns of W, takes the residual stream).
PROJ = (("in_proj", 3 * T_MODEL, T_MODEL, False), ("out_proj", T_MODEL, T_MODEL, True),
        ("linear_in", 2 * T_FFN, T_MODEL, False), ("linear_out", T_MODEL, T_FFN, True))
PRECISIONS = {"f32": sts.PREC_F32, "bf16": sts.PREC_BF16_MFMA, "split": sts.PREC_F32_SPLIT_BF16}
DEPF = dict(temp=0.8, top_k=250, penalty=1.2)  # the engine's usual sampling settings


def listed():
    decode = dict(kind="decode", heads=T_HEADS, kv_heads=T_HEADS, dim=T_DIM, ring=T_RING, batch=1)
    prefill = dict(kind="prefill", heads=T_HEADS, kv_heads=T_HEADS, dim=T_DIM, ring=T_RING)
    return [
        # A long conversation: the ring is full and wrapped, every frame reads all of it.
        dict(decode, name="decode_full_ring", length=3000),
        # The first seconds of a conversation: little to read, latency counts.
        dict(decode, name="decode_early", length=130),
        # A server's 64 concurrent conversations, each of its own age.
        dict(name="ragged_64_streams", kind="ragged", streams=64, heads=T_HEADS, dim=T_DIM,
             ring=T_RING, shortest=128),
        # A system prompt or voice prompt chunk behind an earlier one, bf16 mirror kept.
        dict(prefill, name="prefill_512_bf16", cached=256, rows=512, precision="bf16",
             mirror=True),
        # The same at the reference's own precision, a ragged chunk.
        dict(prefill, name="prefill_300_f32", cached=1100, rows=300, precision="f32",
             mirror=False),
        # A few injected tokens in the middle of a long conversation, f32 caches only.
        dict(prefill, name="prefill_24_bf16", cached=2500, rows=24, precision="bf16",
             mirror=False),
        # One token of one stream through a temporal layer's projections.
        dict(name="proj_1_token", kind="proj", streams=1, rows=1),
        # One token of each of 13 concurrent streams.
        dict(name="proj_13_streams", kind="proj", streams=13, rows=1),
        # A prompt chunk through the projections.
        dict(name="proj_chunk_512", kind="proj", streams=1, rows=512),
        # A frame's audio tokens for one conversation, and for 64 of them.
        dict(name="depformer_1_stream", kind="depformer", streams=1),
        dict(name="depformer_64_streams", kind="depformer", streams=64),
        # The last depth step's attention on its own: a few microseconds.
        dict(name="depstep_64_streams", kind="depstep", streams=64, heads=16, dim=64, ring=9,
             step=7),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "ragged", "prefill", "prefill", "proj", "proj", "depformer",
                       "depstep"])
    if kind == "decode":
        heads, dim = rng.choice([(32, 128), (32, 128), (16, 64)])
        return dict(kind=kind, heads=heads, kv_heads=heads // rng.choice([1, 1, 4]), dim=dim,
                    ring=T_RING, batch=rng.choice([1, 1, 1, 2, 5]), length=_log(rng, 40, 3000))
    if kind == "ragged":
        return dict(kind=kind, streams=_log(rng, 2, 60), heads=T_HEADS, dim=T_DIM,
                    ring=rng.randint(1500, T_RING), shortest=rng.randint(1, 200))
    if kind == "prefill":
        precision = rng.choice(["f32", "bf16", "bf16", "split"])
        rows = _log(rng, 2, 700)
        return dict(kind=kind, heads=T_HEADS, kv_heads=T_HEADS // rng.choice([1, 1, 1, 4]),
                    dim=T_DIM, ring=T_RING, cached=rng.randint(0, 2200), rows=rows,
                    precision=precision, mirror=precision == "bf16" and rng.random() < 0.5)
    if kind == "proj":
        if rng.random() < 0.5:
            return dict(kind=kind, streams=_log(rng, 2, 64), rows=1)
        return dict(kind=kind, streams=1, rows=_log(rng, 2, 500))
    if kind == "depformer":
        return dict(kind=kind, streams=_log(rng, 2, 63))
    return dict(kind=kind, streams=_log(rng, 1, 200), heads=16, dim=64, ring=9,
                step=rng.randint(0, 8))


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 2654435761 % (1 << 62))


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device=DEV)


def _q4k(g, n, k, count=1):
    """`count` Q4_K matrices [n][k] as a quantiser leaves Gaussian weights of
    variance 1/k: per 32 weights a 6-bit scale with the min at 7.5 of its
    steps, quants normal about the middle.  uint8 [count, n*k/256*144]."""
    blocks = count * n * k // 256
    sc = torch.randint(28, 64, (blocks, 8), generator=g, device=DEV, dtype=torch.uint8)
    lo, hi = sc[:, :4], sc[:, 4:]
    top = lo | ((hi >> 4) << 6)  # scale and min of sub-block j < 4 with the high bits of j + 4
    raw = torch.empty((blocks, 144), dtype=torch.uint8, device=DEV)
    # Mean scale 45.5, quant deviation about 2.7: d so that weights come out at 1/sqrt(k).
    d = 1.0 / (math.sqrt(k) * 45.5 * 2.7)
    dm = torch.empty((blocks, 2), device=DEV)
    dm[:, 0] = d * (0.8 + 0.4 * torch.rand(blocks, generator=g, device=DEV))
    dm[:, 1] = 7.5 * dm[:, 0]
    raw[:, :4] = dm.half().view(torch.uint8)
    raw[:, 4:8] = top
    raw[:, 8:12] = top
    raw[:, 12:16] = (hi & 15) | ((hi & 15) << 4)
    for a in range(0, blocks, 1 << 19):
        z = torch.randn((min(1 << 19, blocks - a), 2, 128), generator=g, device=DEV)
        q = z.mul_(2.7).add_(7.5).round_().clamp_(0, 15).to(torch.uint8)
        raw[a:a + q.shape[0], 16:] = q[:, 0] | (q[:, 1] << 4)
    return raw.view(count, -1)


def _q4_0(g, vocab, dim, count=1):
    """Q4_0 embedding tables: f16 scale and 32 nibbles a block."""
    blocks = count * vocab * dim // 32
    raw = torch.randint(0, 256, (blocks, 18), generator=g, device=DEV, dtype=torch.uint8)
    s = 0.02 + 0.03 * torch.rand((blocks, 1), generator=g, device=DEV)
    raw[:, :2] = s.half().view(torch.uint8)
    return raw.view(count, -1)


_SHIFT = 1234  # rows an old conversation has already pushed out of its ring


def _prepare_decode(case, g):
    full = case["length"] == case["ring"]
    b, d = case["batch"], case["dim"]
    c = sts.KVCache(case["ring"], case["kv_heads"], d, n_heads=case["heads"])
    cached = case["length"] if full else case["length"] - 1
    if full:
        c.advance(_SHIFT)  # an old conversation: the write head is mid-ring
    k = _randn(g, b, cached, case["kv_heads"], d)
    v = _randn(g, b, cached, case["kv_heads"], d)
    c.update(k, v)
    return dict(cache=c, rope=sts.RoPE(d, 8192, THETA), q=_randn(g, b, case["heads"], d),
                k_new=_randn(g, b, case["kv_heads"], d), v_new=_randn(g, b, case["kv_heads"], d),
                out=torch.empty((b, case["heads"], d), device=DEV), scale=sts.softmax_scale(d),
                rows=(k, v), pos=c.offset())


def _prepare_prefill(case, g):
    d = case["dim"]
    c = sts.KVCache(case["ring"], case["kv_heads"], d, bf16_mirror=case["mirror"],
                    n_heads=case["heads"])
    k = _randn(g, 1, case["cached"], case["kv_heads"], d)
    v = _randn(g, 1, case["cached"], case["kv_heads"], d)
    if case["cached"]:
        c.update(k, v)
    s = case["rows"]
    return dict(cache=c, rope=sts.RoPE(d, 4096, THETA), q=_randn(g, s, case["heads"], d),
                k_new=_randn(g, s, case["kv_heads"], d), v_new=_randn(g, s, case["kv_heads"], d),
                out=torch.empty((s, case["heads"], d), device=DEV), scale=sts.softmax_scale(d),
                rows=(k, v), pos=c.offset(), precision=PRECISIONS[case["precision"]])


def _prepare_ragged(case, g):
    b, h, m, d = case["streams"], case["heads"], case["ring"], case["dim"]
    lens = torch.randint(case["shortest"], m + 1, (b,), generator=g, device=DEV, dtype=torch.int32)
    starts = torch.randint(0, m, (b,), generator=g, device=DEV, dtype=torch.int32)
    return dict(q=_randn(g, b, h, d), k=_randn(g, b, h, m, d), v=_randn(g, b, h, m, d), lens=lens,
                starts=starts, out=torch.empty((b, h, d), device=DEV), scale=sts.softmax_scale(d))


def _prepare_proj(case, g):
    st = {}
    for name, n, k, res in PROJ:
        st[name] = dict(w=sts.Q4KTensor(_q4k(g, n, k)[0], (n, k)),
                        x=_randn(g, case["streams"], case["rows"], k),
                        res=_randn(g, case["streams"], case["rows"], n) if res else None)
    return st


def _depf_config():
    return sts.DepformerConfig.personaplex()


def _prepare_depformer(case, g):
    c, b = _depf_config(), case["streams"]
    S, L, D, F, V, T = (c.num_steps, c.num_layers, c.dim, c.ffn, c.out_vocab, c.temporal_dim)
    raw = {"input_proj": _q4k(g, D, T, S), "attn_in_proj": _q4k(g, 3 * D, D, L * S),
           "attn_out_proj": _q4k(g, D, D, L * S), "ffn_linear_in": _q4k(g, 2 * F, D, L * S),
           "ffn_linear_out": _q4k(g, D, F, L * S), "output_linear": _q4k(g, V, D, S),
           "audio_emb": _q4_0(g, c.audio_emb_vocab, D, c.num_audio_emb)}
    w = {f: list(t.unbind(0)) for f, t in raw.items()}
    w["norm1_alpha"] = [1 + 0.1 * _randn(g, D) for _ in range(L)]
    w["norm2_alpha"] = [1 + 0.1 * _randn(g, D) for _ in range(L)]
    w["text_emb"] = _q4_0(g, c.text_emb_vocab, D)[0]

    def ints(hi, *shape):
        return torch.randint(0, hi, shape, generator=g, device=DEV, dtype=torch.int32)
    return dict(engine=sts.DepthEngine(c, w, max_batch=b), weights=w, hidden=_randn(g, b, T),
                text=ints(c.text_emb_vocab, b), rand=torch.rand((b, S), generator=g, device=DEV),
                ptok=ints(V, b, S, 30), npen=ints(31, b, S),
                tokens=torch.empty((b, S), dtype=torch.int32, device=DEV),
                logits=torch.empty((S, b, V), device=DEV))


def _prepare_depstep(case, g):
    b, h, m, d = case["streams"], case["heads"], case["ring"], case["dim"]
    return dict(qkv=_randn(g, b, 3, h, d), k=_randn(g, b, h, m, d), v=_randn(g, b, h, m, d),
                out=torch.empty((b, h, d), device=DEV), scale=sts.softmax_scale(d))


_PREPARE = dict(decode=_prepare_decode, ragged=_prepare_ragged, prefill=_prepare_prefill,
                proj=_prepare_proj, depformer=_prepare_depformer, depstep=_prepare_depstep)


def prepare(case, seed):
    st = _PREPARE[case["kind"]](case, _gen(seed))
    if case["kind"] in ("decode", "prefill"):
        del st["rows"]  # the cache holds them
    st["case"] = case
    return st


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------

def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "decode":
        out = st["cache"].decode_step(st["q"], st["k_new"], st["v_new"], st["scale"], st["rope"],
                                      out=st["out"])
        st["cache"].rollback(1)  # counters only: the next pass is the same step again
        return out
    if kind == "prefill":
        out = st["cache"].prefill(st["q"], st["k_new"], st["v_new"], st["scale"], st["precision"],
                                  rope=st["rope"], out=st["out"])
        st["cache"].rollback(case["rows"])
        return out
    if kind == "ragged":
        return sts.decode_ring(st["q"], st["k"], st["v"], st["lens"], st["starts"], st["scale"],
                               out=st["out"])
    if kind == "proj":
        out = {}
        for name, _, _, res in PROJ:
            p = st[name]
            out[name] = (sts.q4k_matmul_with_residual(p["x"], p["w"], p["res"]) if res
                         else sts.q4k_matmul(p["x"], p["w"]))
        return out
    if kind == "depformer":
        st["engine"].generate(st["hidden"], st["text"], DEPF["temp"], DEPF["top_k"],
                              DEPF["penalty"], st["rand"], st["ptok"], st["npen"],
                              tokens=st["tokens"], logits=st["logits"])
        return dict(tokens=st["tokens"], logits=st["logits"])
    x = st["qkv"]
    sts.depformer_step(x[:, 0], x[:, 1], x[:, 2], st["k"], st["v"], case["step"], st["scale"],
                       out=st["out"], qkv_stride=3 * case["heads"] * case["dim"])
    return dict(out=st["out"], k=st["k"], v=st["v"])


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind == "decode":
        b, h, hk, d, n = (case["batch"], case["heads"], case["kv_heads"], case["dim"],
                          case["length"])
        # The new row comes in from k_new / v_new and goes out to the cache.
        return dict(bytes=4 * b * d * (2 * hk * (n + 1) + 2 * h), flops=4 * b * h * d * n)
    if kind == "ragged":
        b, h, d = case["streams"], case["heads"], case["dim"]
        rows = b * (case["shortest"] + case["ring"]) / 2
        return dict(bytes=8 * h * d * (rows + b), flops=4 * h * d * rows)
    if kind == "prefill":
        h, hk, d, s, c = (case["heads"], case["kv_heads"], case["dim"], case["rows"],
                          case["cached"])
        # K/V: the cached rows (from the mirror where there is one), the chunk's
        # rows in and out (the mirror's copy too); q in, out out.
        kv = 2 * hk * d * (c * (2 if case["mirror"] else 4) + s * (10 if case["mirror"] else 8))
        return dict(bytes=kv + 8 * s * h * d, flops=4 * h * d * (s * c + s * (s + 1) // 2))
    if kind == "proj":
        m = case["streams"] * case["rows"]
        return dict(bytes=sum(n * k * 9 // 16 + 4 * m * (k + n * (2 if res else 1))
                              for _, n, k, res in PROJ),
                    flops=sum(2 * m * n * k for _, n, k, _ in PROJ))
    if kind == "depformer":
        c, b = _depf_config(), case["streams"]
        S, L, D, F, V, T = (c.num_steps, c.num_layers, c.dim, c.ffn, c.out_vocab, c.temporal_dim)
        w = S * (D * T + V * D) + L * S * (4 * D * D + 3 * F * D)
        return dict(bytes=w * 9 // 16 + 4 * b * (T + S * V) + S * b * (D * 9 // 16 + 4 * 33),
                    flops=2 * b * w)
    b, h, d, n = case["streams"], case["heads"], case["dim"], case["step"] + 1
    return dict(bytes=4 * b * h * d * (2 * n + 2 + 2), flops=4 * b * h * d * n)


def tolerance(case):
    kind = case["kind"]
    if kind == "depformer":
        # Eight steps of six f32 layers (6e-7 from 64 bits measured); a draw within
        # rounding of a boundary may fall either way.
        return {"rel": 1e-5, "max": 4e-4, "differ": 0.01}
    if kind == "prefill" and case["precision"] == "bf16":
        return {"rel": 1e-2, "max": 0.2}  # 3.3e-3 from 64 bits measured
    if kind == "prefill" and case["precision"] == "split":
        return {"rel": 3e-5, "max": 1e-3}  # 6.4e-6 measured
    return {"rel": 1e-5, "max": 4e-4}


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------

def _rope64(x, pos):
    """x [rows, heads, d] rotated at pos, pos + 1, ...: interleaved pairs, the
    angle taken in f32 as the model takes it, the rest in 64 bits."""
    rows, _, d = x.shape
    j = torch.arange(0, d, 2, dtype=torch.float32)
    inv = (1.0 / torch.pow(torch.tensor(THETA, dtype=torch.float32), j / d)).to(x.device)
    p = torch.arange(pos, pos + rows, dtype=torch.float32, device=x.device)
    ang = (p[:, None] * inv[None]).double()[:, None, :]
    a, b = x[..., 0::2], x[..., 1::2]
    y = torch.empty_like(x)
    y[..., 0::2] = a * ang.cos() - b * ang.sin()
    y[..., 1::2] = a * ang.sin() + b * ang.cos()
    return y


def _attend64(q, k, v, scale, base=None):
    """q [h, s, d], k / v [hk, n, d] -> [h, s, d]; query i sees rows 0..base+i (all if None)."""
    h, s, _ = q.shape
    out = torch.empty_like(q)
    for i in range(h):
        kv = i // (h // k.shape[0])
        w = (q[i] @ k[kv].transpose(0, 1).contiguous()) * scale
        if base is not None:
            row = torch.arange(k.shape[1], device=q.device)
            w.masked_fill_(row[None] > base + torch.arange(s, device=q.device)[:, None],
                           float("-inf"))
        out[i] = w.softmax(-1) @ v[kv]
    return out


def _exact_decode(case, st):
    k, v = (t.double() for t in st["rows"])
    if case["length"] == case["ring"]:
        k, v = k[:, 1:], v[:, 1:]  # the step overwrites the oldest row
    outs = []
    for b in range(case["batch"]):
        q = _rope64(st["q"][b:b + 1].double(), st["pos"])
        kn = _rope64(st["k_new"][b:b + 1].double(), st["pos"])
        kk = torch.cat([k[b], kn]).transpose(0, 1).contiguous()
        vv = torch.cat([v[b], st["v_new"][b:b + 1].double()]).transpose(0, 1).contiguous()
        outs.append(_attend64(q.transpose(0, 1).contiguous(), kk, vv, st["scale"])[:, 0])
    return torch.stack(outs)


def _exact_prefill(case, st):
    k, v = (t[0].double() for t in st["rows"])
    q = _rope64(st["q"].double(), st["pos"]).transpose(0, 1).contiguous()
    kk = torch.cat([k, _rope64(st["k_new"].double(), st["pos"])]).transpose(0, 1).contiguous()
    vv = torch.cat([v, st["v_new"].double()]).transpose(0, 1).contiguous()
    return _attend64(q, kk, vv, st["scale"], base=case["cached"]).transpose(0, 1).contiguous()


def _exact_ragged(case, st):
    out = torch.zeros_like(st["q"], dtype=torch.float64)
    for b, (n, a) in enumerate(zip(st["lens"].tolist(), st["starts"].tolist())):
        if n:
            idx = (a + torch.arange(n, device=DEV)) % case["ring"]
            out[b] = _attend64(st["q"][b].double()[:, None], st["k"][b][:, idx].double(),
                               st["v"][b][:, idx].double(), st["scale"])[:, 0]
    return out


def _dequant64(raw, n, k):
    """Q4_K bytes -> [n, k] weights d*scale*q - dmin*min in 64 bits."""
    r = raw.view(-1, 144)
    dd = r[:, :4].contiguous().view(torch.half).double()
    s = r[:, 4:16].to(torch.int32)
    sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1)
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
    qs = r[:, 16:].view(-1, 4, 1, 32)
    q = torch.cat([qs & 15, qs >> 4], 2).view(-1, 8, 32)
    w = (dd[:, :1] * sc)[..., None] * q - (dd[:, 1:] * mn)[..., None]
    return w.view(n, k)


def _times(x, raw, n, k):
    return x @ _dequant64(raw, n, k).transpose(0, 1)


def _exact_proj(case, st):
    out = {}
    for name, n, k, res in PROJ:
        y = _times(st[name]["x"].double().view(-1, k), st[name]["w"].raw, n, k)
        y = y.view(case["streams"], case["rows"], n)
        out[name] = y + st[name]["res"].double() if res else y
    return out


def _embed64(table, dim, tok):
    r = table.view(-1, dim // 32, 18)[tok.long()]
    s = r[..., :2].contiguous().view(torch.half).double()
    q = torch.cat([r[..., 2:] & 15, r[..., 2:] >> 4], -1).double() - 8
    return (q * s).view(tok.shape[0], dim)


def _sample64(lg, st, s):
    b, V = lg.shape
    listed_ = torch.zeros((b, V + 1), dtype=torch.bool, device=DEV)
    use = torch.arange(30, device=DEV)[None] < st["npen"][:, s, None]
    listed_.scatter_(1, torch.where(use, st["ptok"][:, s], V).long(), True)
    p = DEPF["penalty"]
    x = torch.where(listed_[:, :V], torch.where(lg > 0, lg / p, lg * p), lg) / DEPF["temp"]
    val, idx = x.sort(dim=1, descending=True, stable=True)
    val, idx = val[:, :DEPF["top_k"]], idx[:, :DEPF["top_k"]]
    cum = val.softmax(1).cumsum(1)
    pick = (st["rand"][:, s, None].double() >= cum).sum(1).clamp(max=val.shape[1] - 1)
    return idx.gather(1, pick[:, None])[:, 0]


def _exact_depformer(case, st):
    c, w, b = _depf_config(), st["weights"], case["streams"]
    S, L, D, F, V, T = (c.num_steps, c.num_layers, c.dim, c.ffn, c.out_vocab, c.temporal_dim)
    H, hd = c.num_heads, c.dim // c.num_heads

    def norm(x, alpha):
        return x / (x.square().mean(1, keepdim=True) + c.rms_eps).sqrt() * alpha.double()
    tok, logits, tokens = st["text"], [], []
    past = [([], []) for _ in range(L)]
    for s in range(S):
        table = w["text_emb"] if s == 0 else w["audio_emb"][min(s - 1, c.num_audio_emb - 1)]
        h = _times(st["hidden"].double(), w["input_proj"][s], D, T) + _embed64(table, D, tok)
        for n in range(L):
            i = n * S + s
            qkv = _times(norm(h, w["norm1_alpha"][n]), w["attn_in_proj"][i], 3 * D, D)
            q, k, v = qkv.view(b, 3, H, hd).unbind(1)
            past[n][0].append(k)
            past[n][1].append(v)
            kk, vv = (torch.stack(t, 2) for t in past[n])  # [b, H, s + 1, hd]
            a = ((q[:, :, None] * kk).sum(-1) * c.attn_scale).softmax(-1)
            h = h + _times((a[..., None] * vv).sum(2).view(b, D), w["attn_out_proj"][i], D, D)
            gv = _times(norm(h, w["norm2_alpha"][n]), w["ffn_linear_in"][i], 2 * F, D)
            act = torch.nn.functional.silu(gv[:, :F]) * gv[:, F:]
            h = h + _times(act, w["ffn_linear_out"][i], D, F)
        logits.append(_times(h, w["output_linear"][s], V, D))
        tok = _sample64(logits[-1], st, s)
        tokens.append(tok)
    return dict(tokens=torch.stack(tokens, 1).int(), logits=torch.stack(logits))


def _exact_depstep(case, st):
    n, b = case["step"], case["streams"]
    q, k_new, v_new = (t.double() for t in st["qkv"].unbind(1))
    k, v = st["k"].double(), st["v"].double()
    k[:, :, n], v[:, :, n] = k_new, v_new
    a = ((q[:, :, None] * k[:, :, :n + 1]).sum(-1) * st["scale"]).softmax(-1)
    return dict(out=(a[..., None] * v[:, :, :n + 1]).sum(2).view(b, case["heads"], case["dim"]),
                k=k, v=v)


_EXACT = dict(decode=_exact_decode, ragged=_exact_ragged, prefill=_exact_prefill,
              proj=_exact_proj, depformer=_exact_depformer, depstep=_exact_depstep)


def exact(case, seed):
    return _EXACT[case["kind"]](case, _PREPARE[case["kind"]](case, _gen(seed)))
