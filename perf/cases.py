"""The measured cases: what a serving engine has this library do, tick by tick.

Three kinds of case.
  attn   one engine tick's attention: the step's rows are packed once
         (Context.pack_step) and every layer of the pool is attended
         (Context.attention_step), as the engine loop does it.
  block  one engine tick's attention block: pack, then per layer the Q, K and V
         projections (Context.matmul_batch), RoPE with the KV write
         (Pool.rope_write_step), attention, and the output projection.  Each
         layer has its own input: the norms and the FFN between them are the
         caller's.
  proj   one projection of a batch of activations.
The ragged lengths of a case come from its number "lens"; page placement,
activations, weights and cached K/V come from the seed.
"""
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "glacier.serve_amd"))
import glacier_paged as gsp  # noqa: E402

WTYPES = {"f32": gsp.WTYPE_F32, "q8_0": gsp.WTYPE_Q8_0, "q4_k": gsp.WTYPE_Q4_K, "q6_k": gsp.WTYPE_Q6_K}
BITS = {"f32": 32.0, "q8_0": 34 * 8 / 32, "q4_k": 144 * 8 / 256, "q6_k": 210 * 8 / 256}
FREQ_BASE = 1.0e6
MAX_SEQ = 65536


def _attn(name, heads, kv_heads, head_dim, kv, decode_rows, ctx_lo, ctx_hi, layers, lens, page=16, prefill_rows=0,
          prior_hi=0, chunk_lo=0, chunk_hi=0):
    return {"name": name, "kind": "attn", "heads": heads, "kv_heads": kv_heads, "head_dim": head_dim, "kv": kv,
            "page": page, "decode_rows": decode_rows, "ctx_lo": ctx_lo, "ctx_hi": ctx_hi,
            "prefill_rows": prefill_rows, "prior_hi": prior_hi, "chunk_lo": chunk_lo, "chunk_hi": chunk_hi,
            "layers": layers, "lens": lens}


def _block(name, w_qk, w_v, w_o, **kw):
    c = _attn(name, **kw)
    c.update(kind="block", w_qk=w_qk, w_v=w_v, w_o=w_o)
    return c


def _proj(name, w, rows, in_dim, out_dim):
    return {"name": name, "kind": "proj", "w": w, "rows": rows, "in_dim": in_dim, "out_dim": out_dim}


def listed():
    return [
        # The smallest tick: a small model (14/2 heads, d 64) serving 8 short chats.  Launches and host time.
        _attn("decode_8rows_f32", 14, 2, 64, "f32", 8, 1, 256, 4, 11),
        # The headline decode tick: 28/4 heads, d 128, 64 ragged rows, fp32 pages.
        _attn("decode_64rows_f32", 28, 4, 128, "f32", 64, 128, 4096, 4, 12),
        # A full batch on fp16 pages (32/8 heads), 256 rows of mixed age.
        _attn("decode_256rows_f16", 32, 8, 128, "f16", 256, 64, 8192, 3, 13),
        # Long documents: 64/8 heads, 16 rows of 16k to 32k tokens, fp16 pages.
        _attn("decode_long_f16", 64, 8, 128, "f16", 16, 16384, 32768, 2, 14),
        # Continuous batching proper: 48 decode rows beside 16 ragged prefill chunks, fp32 pages.
        _attn("mixed_f32", 28, 4, 128, "f32", 48, 256, 4096, 2, 15, prefill_rows=16, prior_hi=2048, chunk_lo=32,
              chunk_hi=512),
        # Admission: prompts of ragged length over short cached prefixes, no decode rows, fp16 pages.
        _attn("prefill_f16", 32, 8, 128, "f16", 0, 0, 0, 2, 16, prefill_rows=12, prior_hi=1024, chunk_lo=100,
              chunk_hi=700),
        # A model off the tuned widths: 2/1 heads, d 32, 8-token pages, 256 rows.
        _attn("decode_small_heads_f32", 2, 1, 32, "f32", 256, 128, 4096, 4, 17, page=8),
        # A decode batch's Q (or output) projection with Q8_0 weights.
        _proj("proj_q8_0_64", "q8_0", 64, 3584, 3584),
        # The same batch's widest projection with Q4_K weights.
        _proj("proj_q4_k_64_wide", "q4_k", 64, 3584, 18944),
        # A prefill chunk's projection with Q6_K weights, an odd number of rows.
        _proj("proj_q6_k_1019", "q6_k", 1019, 3584, 3584),
        # Unquantized weights under a 256-row batch.
        _proj("proj_f32_256", "f32", 256, 4096, 4096),
        # The whole attention block of a decode tick with the usual 4-bit mix (V in 6 bits).
        _block("block_64rows_q4_k", "q4_k", "q6_k", "q4_k", heads=28, kv_heads=4, head_dim=128, kv="f32",
               decode_rows=64, ctx_lo=128, ctx_hi=2048, layers=2, lens=18),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ranges; it costs no more than decode_256rows_f16 in bytes or mixed_f32 in operations."""
    lens = rng.randrange(1 << 30)
    pick = rng.random()
    if pick < 0.4:
        w = rng.choice(["f32", "q8_0", "q4_k", "q6_k"])
        in_dim = 256 * _log_int(rng, 2, 74) if w.endswith("_k") else 64 * _log_int(rng, 8, 296)
        out_dim = _log_int(rng, 256, 32768)
        rows = min(_log_int(rng, 1, 4096), max(1, int(60e9 / (2 * in_dim * out_dim))))
        if out_dim % 16 == 0:
            out_dim += rng.choice([0, 0, 4, 1])
        c = _proj("", w, rows, in_dim, out_dim)
    else:
        heads, kv_heads, head_dim, page = rng.choice([(14, 2, 64, 16), (28, 4, 128, 16), (32, 8, 128, 16),
                                                      (64, 8, 128, 16), (2, 1, 32, 8)])
        kv = rng.choice(["f32", "f16"])
        elem = 4 if kv == "f32" else 2
        layers = rng.choice([1, 2, 4])
        per_token = 2 * kv_heads * head_dim * elem * layers
        block = pick > 0.85 and head_dim >= 64
        prefill = pick > 0.6 and head_dim >= 64
        hi = _log_int(rng, 256, 8192 if prefill or block else 32768)
        lo = _log_int(rng, 1, hi)
        rows = max(1, min(_log_int(rng, 1, 256), int(3.5e9 / (per_token * hi))))
        kw = dict(decode_rows=rows, ctx_lo=lo, ctx_hi=hi, layers=layers, lens=lens, page=page)
        if prefill:
            chunk = _log_int(rng, 2, 512)
            wide = heads * head_dim
            per_query = layers * wide * (4 * 1500 + (5 * wide if block else 0))
            chunk = max(2, min(chunk, int(100e9 / per_query)))
            n = max(1, min(_log_int(rng, 1, 16), int(100e9 / (per_query * chunk))))
            kw.update(prefill_rows=n, prior_hi=rng.choice([0, 500, 2048]), chunk_lo=max(1, chunk // 8), chunk_hi=chunk,
                      decode_rows=rng.choice([0, rows]))
        if block:
            quants = ["q8_0"] if heads * head_dim % 256 else ["q8_0", "q4_k", "q6_k"]
            w = [rng.choice(quants) for _ in range(3)]
            c = _block("", *w, heads=heads, kv_heads=kv_heads, head_dim=head_dim, kv=kv, **kw)
        else:
            c = _attn("", heads, kv_heads, head_dim, kv, **kw)
    del c["name"]
    return c


# ---- what a program has in hand ---------------------------------------------

_CTX = None


def _context():
    """The engine's one context, on a stream of its own."""
    global _CTX
    if _CTX is None:
        _CTX = gsp.Context(0)
    return _CTX


def _rows(case):
    """(tokens before the step, query tokens) of each row."""
    rng = np.random.default_rng(case["lens"])
    n = case["decode_rows"]
    if n:
        lo, hi = math.log(case["ctx_lo"]), math.log(case["ctx_hi"])
        ctx = np.rint(np.exp(rng.uniform(lo, hi, n))).astype(np.int64)
    else:
        ctx = np.zeros(0, np.int64)
    m = case["prefill_rows"]
    prior = rng.integers(0, case["prior_hi"] + 1, m)
    chunk = rng.integers(case["chunk_lo"], case["chunk_hi"] + 1, m)
    return np.concatenate([ctx - 1, prior]), np.concatenate([np.ones(n, np.int64), chunk])


class _Step:
    """A step's packed tables: every row's pages drawn from a pool with a fifth to spare."""

    def __init__(self, case, seed):
        prior, q_lens = _rows(case)
        total = prior + q_lens
        pages = -(-total // case["page"])
        rng = np.random.default_rng([case["lens"], seed])
        self.blocks = int(pages.sum()) * 6 // 5 + 1
        self.positions = prior.astype(np.int32)
        self.q_lens = q_lens.astype(np.int32)
        self.tokens = total.astype(np.int32)
        self.offsets = np.concatenate([[0], np.cumsum(pages)]).astype(np.int32)
        self.ids = rng.permutation(self.blocks)[: int(pages.sum())].astype(np.int32)
        self.total_q = int(q_lens.sum())


class _State:
    """Device buffers and, for a step, the pool over the caller's own arenas."""

    def __init__(self, case):
        self.case = case
        self.pool = None

    def __del__(self):
        if self.pool is not None:
            self.pool.destroy()


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _normal(shape, g, dtype=torch.float32):
    if dtype == torch.float32:
        return torch.randn(shape, generator=g, device="cuda")
    out = torch.empty(shape, device="cuda", dtype=dtype)
    for part in out.view(shape[0], -1).split(4096):
        part.copy_(torch.randn(part.shape, generator=g, device="cuda"))
    return out


def _activations(rows, dim, g):
    """Normed activations: unit scale with a few channels an order of magnitude larger."""
    x = torch.randn((rows, dim), generator=g, device="cuda")
    loud = torch.rand((dim,), generator=g, device="cuda") < 0.005
    return x * torch.where(loud, 12.0, 1.0)


def _le16(t):
    return t.to(torch.float16).contiguous().view(torch.uint8)


def _encode(w_type, w):
    """Rows of fp32 weights in the GGUF layout of `w_type`, rounded to its grid."""
    n, k = w.shape
    if w_type == "f32":
        return w.contiguous()
    if w_type == "q8_0":
        b = w.view(n, k // 32, 32)
        d = (b.abs().amax(-1, keepdim=True) / 127).to(torch.float16)
        q = torch.clamp(torch.round(b / d.float()), -127, 127).to(torch.int8).view(torch.uint8)
        return torch.cat([_le16(d), q], -1).reshape(n, -1).contiguous()
    if w_type == "q4_k":
        b = w.view(n, k // 256, 8, 32)
        lo = torch.clamp(b.amin(-1), max=0.0)
        step = (b.amax(-1) - lo) / 15
        d = (step.amax(-1, keepdim=True) / 63).to(torch.float16)
        dmin = (-lo.amin(-1, keepdim=True) / 63).to(torch.float16)
        sc = torch.clamp(torch.round(step / d.float()), 1, 63)
        m = torch.clamp(torch.round(-lo / dmin.float()), 0, 63)
        q = torch.round((b + (dmin.float() * m).unsqueeze(-1)) / (d.float() * sc).unsqueeze(-1))
        q = torch.clamp(q, 0, 15).to(torch.uint8)
        sc, m = sc.to(torch.uint8), m.to(torch.uint8)
        head = [sc[..., :4] | (sc[..., 4:] >> 4 << 6), m[..., :4] | (m[..., 4:] >> 4 << 6),
                (sc[..., 4:] & 15) | (m[..., 4:] & 15) << 4]
        qs = (q[..., 0::2, :] | q[..., 1::2, :] << 4).reshape(n, k // 256, 128)
        return torch.cat([_le16(d), _le16(dmin), *head, qs], -1).reshape(n, -1).contiguous()
    b = w.view(n, k // 256, 16, 16)
    step = b.abs().amax(-1) / 31
    d = (step.amax(-1, keepdim=True) / 127).to(torch.float16)
    sc = torch.clamp(torch.round(step / d.float()), 1, 127)
    q = torch.clamp(torch.round(b / (d.float() * sc).unsqueeze(-1)), -32, 31) + 32
    q = q.to(torch.uint8).view(n, k // 256, 2, 4, 32)  # halves of four 32-wide quarters
    ql = torch.cat([(q[..., :2, :] & 15) | (q[..., 2:, :] & 15) << 4], -2).reshape(n, k // 256, 128)
    h = q >> 4
    qh = (h[..., 0, :] | h[..., 1, :] << 2 | h[..., 2, :] << 4 | h[..., 3, :] << 6).reshape(n, k // 256, 64)
    return torch.cat([ql, qh, sc.to(torch.int8).view(torch.uint8), _le16(d)], -1).reshape(n, -1).contiguous()


def _half(b):
    return b.contiguous().view(torch.float16).double()


def _decode(w_type, raw, in_dim):
    """The float64 weights that rows of `w_type` stand for."""
    n = raw.shape[0]
    if w_type == "f32":
        return raw.double()
    if w_type == "q8_0":
        b = raw.view(n, in_dim // 32, 34)
        return (_half(b[..., :2]) * b[..., 2:].contiguous().view(torch.int8).double()).reshape(n, in_dim)
    if w_type == "q4_k":
        b = raw.view(n, in_dim // 256, 144)
        d, dmin = _half(b[..., 0:2]), _half(b[..., 2:4])
        s0, s1, s2 = b[..., 4:8], b[..., 8:12], b[..., 12:16]
        sc = torch.cat([s0 & 63, (s2 & 15) | (s0 >> 6 << 4)], -1).double()
        m = torch.cat([s1 & 63, (s2 >> 4) | (s1 >> 6 << 4)], -1).double()
        qs = b[..., 16:].reshape(n, -1, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], -2).reshape(n, -1, 8, 32).double()
        return ((d * sc).unsqueeze(-1) * q - (dmin * m).unsqueeze(-1)).reshape(n, in_dim)
    b = raw.view(n, in_dim // 256, 210)
    ql = b[..., :128].reshape(n, -1, 2, 2, 32)
    qh = b[..., 128:192].reshape(n, -1, 2, 32)
    low = torch.cat([ql & 15, ql >> 4], -2)
    high = torch.stack([qh & 3, (qh >> 2) & 3, (qh >> 4) & 3, qh >> 6], -2)
    q = (low | high << 4).reshape(n, -1, 16, 16).double() - 32
    sc = b[..., 192:208].contiguous().view(torch.int8).double()
    return ((_half(b[..., 208:]) * sc).unsqueeze(-1) * q).reshape(n, in_dim)


def _weights(w_type, out_dim, in_dim, g):
    w = torch.empty((out_dim, in_dim), device="cuda")
    w.normal_(0.0, 1.0 / math.sqrt(in_dim), generator=g)
    return _encode(w_type, w)


def prepare(case, seed):
    s = _State(case)
    g = _gen(seed)
    s.ctx = _context()
    if case["kind"] == "proj":
        s.w = _weights(case["w"], case["out_dim"], case["in_dim"], g)
        s.x = _activations(case["rows"], case["in_dim"], g)
        s.y = torch.zeros((case["rows"], case["out_dim"]), device="cuda")
        torch.cuda.synchronize()
        return s
    s.step = step = _Step(case, seed)
    heads, kvh, d, layers = case["heads"], case["kv_heads"], case["head_dim"], case["layers"]
    dtype = torch.float32 if case["kv"] == "f32" else torch.float16
    shape = (step.blocks, layers, kvh, case["page"], d)
    s.k, s.v = _normal(shape, g, dtype), _normal(shape, g, dtype)
    s.pool = gsp.Pool.wrap(s.ctx, s.k.data_ptr(), s.v.data_ptr(), step.blocks, layers, kvh, d,
                           gsp.KV_F32 if case["kv"] == "f32" else gsp.KV_F16, block_size=case["page"])
    s.scale = 1.0 / math.sqrt(d)
    s.out = [torch.zeros((step.total_q, heads, d), device="cuda") for _ in range(layers)]
    if case["kind"] == "attn":
        s.q = [torch.randn((step.total_q, heads, d), generator=g, device="cuda") for _ in range(layers)]
    else:
        hidden = heads * d
        types = (case["w_qk"], case["w_qk"], case["w_v"], case["w_o"])
        outs = (hidden, kvh * d, kvh * d, hidden)
        s.w = [[_weights(t, o, hidden, g) for t, o in zip(types, outs)] for _ in range(layers)]
        s.x = [_activations(step.total_q, hidden, g) for _ in range(layers)]
        s.q = [torch.zeros((step.total_q, heads, d), device="cuda") for _ in range(layers)]
        s.kn = [torch.zeros((step.total_q, kvh, d), device="cuda") for _ in range(layers)]
        s.vn = [torch.zeros((step.total_q, kvh, d), device="cuda") for _ in range(layers)]
        s.y = [torch.zeros((step.total_q, hidden), device="cuda") for _ in range(layers)]
    torch.cuda.synchronize()
    return s


def run(s):
    case, ctx = s.case, s.ctx
    if case["kind"] == "proj":
        ctx.matmul_batch(WTYPES[case["w"]], s.w.data_ptr(), s.x.data_ptr(), s.y.data_ptr(), case["in_dim"],
                         case["out_dim"], case["rows"])
        return s.y
    step, heads = s.step, case["heads"]
    ctx.pack_step(s.pool, step.positions, step.tokens, step.offsets, step.ids, MAX_SEQ, q_lens=step.q_lens,
                  want_info=False)
    if case["kind"] == "attn":
        for i in range(case["layers"]):
            ctx.attention_step(s.pool, i, heads, s.q[i].data_ptr(), s.out[i].data_ptr(), s.scale)
        return s.out
    n, hidden, kv_dim = step.total_q, heads * case["head_dim"], case["kv_heads"] * case["head_dim"]
    qk, wv, wo = WTYPES[case["w_qk"]], WTYPES[case["w_v"]], WTYPES[case["w_o"]]
    for i in range(case["layers"]):
        w, x = s.w[i], s.x[i].data_ptr()
        q, k, v, out = s.q[i].data_ptr(), s.kn[i].data_ptr(), s.vn[i].data_ptr(), s.out[i].data_ptr()
        ctx.matmul_batch(qk, w[0].data_ptr(), x, q, hidden, hidden, n)
        ctx.matmul_batch(qk, w[1].data_ptr(), x, k, hidden, kv_dim, n)
        ctx.matmul_batch(wv, w[2].data_ptr(), x, v, hidden, kv_dim, n)
        s.pool.rope_write_step(i, heads, FREQ_BASE, gsp.ROPE_HALVES, q, k, v)
        ctx.attention_step(s.pool, i, heads, q, out, s.scale)
        ctx.matmul_batch(wo, w[3].data_ptr(), out, s.y[i].data_ptr(), hidden, hidden, n)
    return {"y": s.y, "q": s.q, "keys": s.k, "values": s.v}


# ---- what a pass cannot do without -------------------------------------------

def _attn_work(case):
    prior, q_lens = _rows(case)
    tokens = int((prior + q_lens).sum())
    pairs = int((q_lens * prior + q_lens * (q_lens + 1) // 2).sum())
    elem = 4 if case["kv"] == "f32" else 2
    wide = case["heads"] * case["head_dim"]
    return (tokens * 2 * case["kv_heads"] * case["head_dim"] * elem, 4 * wide * pairs, int(q_lens.sum()), wide)


def work(case):
    if case["kind"] == "proj":
        b, i, o = case["rows"], case["in_dim"], case["out_dim"]
        return {"bytes": i * o * BITS[case["w"]] / 8 + 4 * b * (i + o), "flops": 2 * b * i * o}
    kv, flops, n, wide = _attn_work(case)
    if case["kind"] == "attn":
        return {"bytes": case["layers"] * (kv + 8 * n * wide), "flops": case["layers"] * flops}
    kv_dim = case["kv_heads"] * case["head_dim"]
    w = wide * (wide * (BITS[case["w_qk"]] + BITS[case["w_o"]]) + kv_dim * (BITS[case["w_qk"]] + BITS[case["w_v"]])) / 8
    # x in, q and y out, the new K and V into their slots
    acts = 4 * n * 3 * wide + 2 * n * kv_dim * (4 if case["kv"] == "f32" else 2)
    mm = 2 * n * wide * (2 * wide + 2 * kv_dim)
    return {"bytes": case["layers"] * (kv + w + acts), "flops": case["layers"] * (flops + mm)}


def tolerance(case):
    """Sums are 32-bit throughout (measured against float64: 5e-8 to 8e-7); a block on fp16 pages rounds its new keys
    and values to 11 bits, where a last-bit difference before the rounding can move one to its neighbour."""
    if case["kind"] == "block":
        return {"rel": 2e-3, "max": 2e-2} if case["kv"] == "f16" else {"rel": 4e-6, "max": 1e-4}
    return {"rel": 2e-6, "max": 4e-5}


# ---- the same in 64 bits -----------------------------------------------------

def _attend64(case, step, q, k, v):
    """Causal attention of every row over its pages; q [tokens, heads, d] and the layer's arenas [blocks, kv, page, d]."""
    kvh, d = case["kv_heads"], case["head_dim"]
    group = case["heads"] // kvh
    out = torch.zeros(q.shape, dtype=torch.float64, device="cuda")
    at = 0
    for b in range(len(step.positions)):
        pos, ql, total = int(step.positions[b]), int(step.q_lens[b]), int(step.tokens[b])
        ids = torch.from_numpy(step.ids[step.offsets[b]: step.offsets[b + 1]].astype(np.int64)).cuda()
        kk = k[ids].double().transpose(1, 2).reshape(-1, kvh, d)[:total]
        vv = v[ids].double().transpose(1, 2).reshape(-1, kvh, d)[:total]
        for h in range(kvh):
            qq = q[at: at + ql, h * group: (h + 1) * group].double().reshape(ql * group, d)
            sc = torch.matmul(qq, kk[:, h].t().contiguous()) / math.sqrt(d)
            if ql > 1:
                last = pos + torch.arange(ql, device="cuda").repeat_interleave(group)
                sc.masked_fill_(torch.arange(total, device="cuda")[None, :] > last[:, None], -math.inf)
            o = torch.matmul(torch.softmax(sc, -1), vv[:, h].contiguous())
            out[at: at + ql, h * group: (h + 1) * group] = o.view(ql, group, d)
        at += ql
    return out


def _rope64(x, pos):
    half = x.shape[-1] // 2
    rate = FREQ_BASE ** (-torch.arange(half, dtype=torch.float64, device="cuda") / half)
    angle = pos[:, None] * rate
    c, sn = torch.cos(angle)[:, None], torch.sin(angle)[:, None]
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * c - b * sn, a * sn + b * c], -1)


def exact(case, seed):
    s = prepare(case, seed)
    if case["kind"] == "proj":
        return torch.matmul(s.x.double(), _decode(case["w"], s.w, case["in_dim"]).t().contiguous())
    step = s.step
    if case["kind"] == "attn":
        return [_attend64(case, step, s.q[i], s.k[:, i], s.v[:, i]) for i in range(case["layers"])]
    heads, kvh, d, page = case["heads"], case["kv_heads"], case["head_dim"], case["page"]
    hidden = heads * d
    pos = np.concatenate([p + np.arange(n) for p, n in zip(step.positions, step.q_lens)])
    row = np.repeat(np.arange(len(step.positions)), step.q_lens)
    block = torch.from_numpy(step.ids[step.offsets[row] + pos // page].astype(np.int64)).cuda()
    slot = torch.from_numpy(pos % page).cuda()
    at = torch.from_numpy(pos).cuda().double()
    types = (case["w_qk"], case["w_qk"], case["w_v"], case["w_o"])
    got = {"y": [], "q": [], "keys": s.k.double(), "values": s.v.double()}
    for i in range(case["layers"]):
        wq, wk, wv, wo = (_decode(t, w, hidden).t().contiguous() for t, w in zip(types, s.w[i]))
        x = s.x[i].double()
        q = _rope64(torch.matmul(x, wq).view(-1, heads, d), at)
        k = _rope64(torch.matmul(x, wk).view(-1, kvh, d), at)
        v = torch.matmul(x, wv).view(-1, kvh, d)
        if case["kv"] == "f16":
            k, v = k.half().double(), v.half().double()
        got["keys"][:, i][block, :, slot] = k
        got["values"][:, i][block, :, slot] = v
        o = _attend64(case, step, q, got["keys"][:, i], got["values"][:, i])
        got["q"].append(q)
        got["y"].append(torch.matmul(o.view(-1, hidden), wo))
    return got
