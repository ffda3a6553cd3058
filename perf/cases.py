"""The work this package is measured on: the paged KV-cache operators and the decoder
built on them, called as a serving program calls them.

Kinds of cases (field ``kind``):
  decode     one decode step of one attention layer: the new token's K/V rows are appended
             and attended with the cached ones (``paged_decode_append_attention``), or, with
             ``window``, attention over a resident sliding window (``paged_decode_attention``)
  prefill    causal attention of chunks of new tokens over their pages
             (``paged_prefill_attention``)
  append     rows of several chunks scattered into their pages (``kv_append``)
  gather     pages back into contiguous, zero-padded K and V (``kv_gather``)
  roundtrip  an append of whole sequences followed by their gather
  block      one pre-norm transformer block on a batch of prompts, without a cache
  loop       a decoder's prompt forward followed by single-token steps through its cache

Sequence lengths are a function of the case alone; the seed draws the values, the order of
the lengths and the page permutation.  ``exact`` evaluates the same inputs in float64 with
plain torch.
"""
from __future__ import annotations

import math
import random
from statistics import NormalDist

import torch

from __graft_entry__ import load_package

iva = load_package()

BS = 16
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
FP8 = torch.float8_e4m3fn


# ------------------------------------------------------------------------- cases

def listed():
    return [
        # Append and gather of four short fp32 sequences (17 .. 200 tokens, 8 kv heads of
        # 64): the smallest use of the cache, two launches.
        dict(name="roundtrip-4", kind="roundtrip", dtype="fp32", pages="fp32", batch=4, dist="uniform",
             lo=17, hi=200, hkv=8, dim=64),
        # One user's interactive decode step: a single sequence of a short chat.
        dict(name="decode-1", kind="decode", dtype="fp16", pages="fp16", batch=1, dist="uniform", lo=777,
             hi=777, hq=32, hkv=8, dim=128, window=0, sinks=0),
        # The ordinary serving batch: 32 sequences of 512 .. 4096 tokens, GQA 32/8.
        dict(name="decode-32", kind="decode", dtype="fp16", pages="fp16", batch=32, dist="uniform", lo=512,
             hi=4096, hq=32, hkv=8, dim=128, window=0, sinks=0),
        # The same batch on FP8 pages, bf16 model.
        dict(name="decode-32-fp8", kind="decode", dtype="bf16", pages="fp8", batch=32, dist="uniform",
             lo=512, hi=4096, hq=32, hkv=8, dim=128, window=0, sinks=0),
        # Long documents under a sliding window of 4096 with 4 sink tokens, window resident.
        dict(name="decode-window-4", kind="decode", dtype="bf16", pages="bf16", batch=4, dist="uniform",
             lo=32768, hi=131072, hq=32, hkv=8, dim=128, window=4096, sinks=4),
        # A continuous-batching step's decode tokens: 256 ragged sequences (log-normal).
        dict(name="decode-256", kind="decode", dtype="fp16", pages="fp16", batch=256, dist="lognormal",
             lo=1, hi=16384, hq=32, hkv=8, dim=128, window=0, sinks=0),
        # Chunked prefill of 16 prompts in step: 512 new tokens each on 1536 cached.
        dict(name="prefill-16x512", kind="prefill", dtype="fp16", pages="fp16", batch=16, dist="uniform",
             lo=2048, hi=2048, chunk=512, odd=False, hq=32, hkv=8, dim=128, window=0, sinks=0),
        # A continuous-batching step's prefill chunks: 11 sequences at ragged points of
        # prompts up to 8k, the last chunk of a prompt shorter than the others.
        dict(name="prefill-ragged-11", kind="prefill", dtype="bf16", pages="bf16", batch=11, dist="uniform",
             lo=301, hi=8111, chunk=512, odd=True, hq=32, hkv=8, dim=128, window=0, sinks=0),
        # The same step's append: its chunks start wherever the sequences stand.
        dict(name="append-ragged-11", kind="append", dtype="bf16", pages="bf16", batch=11, dist="uniform",
             lo=301, hi=8111, chunk=512, odd=True, hkv=8, dim=128),
        # The serving batch handed to code that wants contiguous K and V.
        dict(name="gather-32", kind="gather", dtype="fp16", pages="fp16", batch=32, dist="uniform", lo=512,
             hi=4096, hkv=8, dim=128),
        # One block of the dense decoder (d_model 1024, 16 heads) on 16 prompts of 512.
        dict(name="block-16x512", kind="block", dtype="bf16", batch=16, tokens=512, d_model=1024, heads=16,
             kv_heads=16),
        # The dense decoder (16 layers, vocabulary 32000): 16 prompts of 512 tokens, then
        # eight single-token steps.
        dict(name="loop-16x512+8", kind="loop", dtype="bf16", batch=16, tokens=512, steps=8, d_model=1024,
             heads=16, kv_heads=16, layers=16, vocab=32000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


_HEADS = [(32, 8), (32, 8), (16, 16), (32, 32), (8, 1), (16, 4), (12, 4)]


def draw(rng: random.Random):
    while True:
        kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "append", "gather", "roundtrip",
                           "block", "loop"])
        dtype = rng.choice(["fp16", "bf16", "bf16", "fp32"] if kind not in ("block", "loop") else ["bf16"])
        if kind in ("block", "loop"):
            d_model, heads, kv_heads = rng.choice([(1024, 16, 16), (512, 8, 2), (256, 4, 2), (1024, 16, 4)])
            c = dict(kind=kind, dtype=dtype, batch=_log_int(rng, 1, 16), tokens=_log_int(rng, 2, 512),
                     d_model=d_model, heads=heads, kv_heads=kv_heads)
            if kind == "loop":
                c.update(steps=rng.randint(1, 8), layers=rng.choice([1, 2, 8, 16]), vocab=rng.choice([512, 32000]))
            return c
        hq, hkv = rng.choice(_HEADS)
        c = dict(kind=kind, dtype=dtype, pages=dtype, batch=_log_int(rng, 1, 256), dist="uniform",
                 lo=1, hi=1, hkv=hkv, dim=rng.choice([64, 128, 128, 256]))
        hi = _log_int(rng, 32, 16384)
        c.update(lo=_log_int(rng, 16, hi), hi=hi)
        if dtype != "fp32" and kind != "roundtrip" and rng.random() < 0.25:
            c.update(pages="fp8")
        if kind in ("decode", "prefill"):
            c.update(hq=hq, window=0, sinks=0)
            if rng.random() < 0.2:
                c.update(window=_log_int(rng, 64, 4096), sinks=rng.choice([0, 4]))
        if kind in ("prefill", "append"):
            c.update(chunk=_log_int(rng, 2, 512), odd=rng.random() < 0.7)
        # no larger than the listed cases of the same kind
        kv = sum(_lengths(c)) * hkv * c["dim"] * 2 * (4 if dtype == "fp32" else 2)
        w = work(c)
        if kv > 2 << 30 or w["bytes"] > 1.7e9 or w["flops"] > (2.4e11 if dtype != "fp32" else 3e10):
            continue
        return c


# ----------------------------------------------------------------------- geometry

def _lengths(c):
    """Context lengths of the case's sequences, ascending: quantiles of its distribution."""
    n = c["batch"]
    if c["dist"] == "lognormal":
        z = [NormalDist().inv_cdf((i + 0.5) / n) for i in range(n)]
        return [max(c["lo"], min(c["hi"], round(1024 * math.exp(x)))) for x in z]
    if n == 1:
        return [c["hi"]]
    return [round(c["lo"] + (c["hi"] - c["lo"]) * i / (n - 1)) for i in range(n)]


def _chunks(c, lengths):
    """New tokens of each sequence: the chunk, or what a prompt's last chunk has left."""
    out = []
    for i, n in enumerate(lengths):
        m = min(c["chunk"], n)
        if c["odd"] and i % 3 == 2:
            m = max(1, min(n, (m * (i % 7 + 1)) // 8 + 1))
        out.append(m)
    return out


def _pairs(c, lengths, chunks):
    """(query row, visible key) pairs of one head."""
    total = 0
    for n, m in zip(lengths, chunks):
        for p in range(n - m, n):
            total += min(p + 1, c["window"] + c["sinks"]) if c["window"] else p + 1
    return total


def _gen(seed, i):
    return torch.Generator(device="cuda").manual_seed((seed * 1000003 + i) % (1 << 62))


def _randn(shape, seed, i, dtype):
    return torch.randn(shape, generator=_gen(seed, i), device="cuda", dtype=dtype)


def _layout(c, seed):
    """(lengths, block table [B, max_blocks] on the host, pages): the lengths in seeded
    order on a seeded permutation of the pool's pages; under a window only the sink pages
    and the window's are resident."""
    r = random.Random(seed)
    lengths = _lengths(c)
    r.shuffle(lengths)
    keep = []
    for n in lengths:
        blocks = -(-n // BS)
        first = max((n - c["window"]) // BS, 0) if c.get("window") and c["kind"] == "decode" else 0
        sinks = -(-c.get("sinks", 0) // BS)
        keep.append([j for j in range(blocks) if j >= first or j < sinks])
    pages = sum(map(len, keep))
    perm = list(range(pages))
    r.shuffle(perm)
    table = torch.full((len(lengths), max(max(k) for k in keep) + 1), -1, dtype=torch.int32)
    at = 0
    for b, k in enumerate(keep):
        table[b, k] = torch.tensor(perm[at:at + len(k)], dtype=torch.int32)
        at += len(k)
    return lengths, keep, table, pages


def _slots(table, b, positions):
    return table[b].long()[positions // BS] * BS + positions % BS


def _resident(keep, length):
    """Positions of a sequence that lie on its resident pages."""
    pos = (torch.tensor(keep, dtype=torch.long)[:, None] * BS + torch.arange(BS)).reshape(-1)
    return pos[pos < length]


def _rows(c, seed, n):
    shape, dt = (n, c["hkv"], c["dim"]), DTYPES[c["dtype"]]
    return _randn(shape, seed, 1, dt), _randn(shape, seed, 2, dt)


def _pools(c, pages):
    dt = FP8 if c["pages"] == "fp8" else DTYPES[c["pages"]]
    ks, vs = iva.pool_shapes(pages, c["hkv"], c["dim"], BS, dt)
    pools = [torch.zeros(ks, dtype=dt, device="cuda"), torch.zeros(vs, dtype=dt, device="cuda")]
    kw = {}
    if dt == FP8:
        shape = iva.scale_shape(pages, c["hkv"], BS)
        kw = {"k_scale": torch.ones(shape, device="cuda"), "v_scale": torch.ones(shape, device="cuda")}
    return pools[0], pools[1], kw


def _state_of(s):
    """The pools as outputs (FP8 codes as bytes, with their factors)."""
    k, v = s["k_pool"], s["v_pool"]
    if k.dtype == FP8:
        return [k.view(torch.uint8), v.view(torch.uint8), s["kw"]["k_scale"], s["kw"]["v_scale"]]
    return [k, v]


def _model(c, seed):
    cfg = iva.TransformerConfig(d_model=c["d_model"], n_heads=c["heads"], n_kv_heads=c["kv_heads"],
                                n_layers=c.get("layers", 1), vocab_size=c.get("vocab", 32), seq_len=1024,
                                dropout=0.0, attn_impl="hip_paged")
    torch.manual_seed(seed)
    with torch.device("cuda"):
        model = iva.Transformer(cfg)
    return model.to(torch.bfloat16).eval()


# ------------------------------------------------------------------- prepare, run

def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "block":
        return dict(kind=kind, block=_model(c, seed).blocks[0],
                    x=_randn((c["batch"], c["tokens"], c["d_model"]), seed, 3, torch.bfloat16))
    if kind == "loop":
        ids = torch.randint(0, c["vocab"], (c["batch"], c["tokens"] + c["steps"]), generator=_gen(seed, 3),
                            device="cuda")
        return dict(kind=kind, model=_model(c, seed), prompt=ids[:, :c["tokens"]].contiguous(),
                    given=ids[:, c["tokens"]:].contiguous())
    lengths, keep, table, pages = _layout(c, seed)
    k_pool, v_pool, kw = _pools(c, pages)
    s = dict(kind=kind, k_pool=k_pool, v_pool=v_pool, kw=kw, tables=table.cuda(),
             lens=torch.tensor(lengths, dtype=torch.int32, device="cuda"))
    resident = [_resident(k, n) for k, n in zip(keep, lengths)]
    slots = torch.cat([_slots(table, b, p) for b, p in enumerate(resident)]).to(torch.int32).cuda()
    k, v = _rows(c, seed, len(slots))
    dt = DTYPES[c["dtype"]]
    if kind in ("roundtrip", "append"):
        if kind == "append":
            new = _new_rows(c, resident, lengths).cuda()
            k, v, slots = k[new], v[new], slots[new]
        s.update(k=k, v=v, slots=slots, out_len=max(lengths))
        return s
    iva.kv_append(k, v, k_pool, v_pool, slots, **kw)
    if kind == "gather":
        s.update(out_len=max(lengths), out_dtype=dt)
    elif kind == "decode":
        s.update(q=_randn((c["batch"], c["hq"], c["dim"]), seed, 4, dt), window=c["window"], sinks=c["sinks"])
        if not c["window"]:
            last = torch.tensor([len(p) for p in resident]).cumsum(0) - 1
            s.update(k=k[last.cuda()], v=v[last.cuda()])
    else:
        chunks = _chunks_of(c, lengths)
        start = torch.tensor([0] + chunks).cumsum(0).to(torch.int32).cuda()
        s.update(q=_randn((sum(chunks), c["hq"], c["dim"]), seed, 4, dt), start=start, longest=max(chunks),
                 window=c["window"], sinks=c["sinks"])
    return s


def _chunks_of(c, lengths):
    """The chunk of each sequence, in the layout's order (equal lengths have equal rank)."""
    left = {}
    for n, m in zip(_lengths(c), _chunks(c, _lengths(c))):
        left.setdefault(n, []).append(m)
    return [left[n].pop(0) for n in lengths]


def _new_rows(c, resident, lengths):
    """Indexes of the chunks' rows among all rows."""
    out, at = [], 0
    for p, n, m in zip(resident, lengths, _chunks_of(c, lengths)):
        out.append(torch.arange(at + n - m, at + n))
        at += len(p)
    return torch.cat(out)


def run(s):
    kind = s["kind"]
    if kind == "block":
        with torch.no_grad():
            return s["block"](s["x"])[0]
    if kind == "loop":
        model, prompt, given = s["model"], s["prompt"], s["given"]
        with torch.no_grad():
            cache = model.new_kv_cache(prompt.shape[0], prompt.shape[1] + given.shape[1])
            logits = [model(prompt, kv_cache=cache)["logits"][:, -1]]
            for t in range(given.shape[1]):
                logits.append(model(given[:, t:t + 1], kv_cache=cache)["logits"][:, -1])
            cache.free()
            return torch.stack(logits, dim=1)
    if kind == "append":
        iva.kv_append(s["k"], s["v"], s["k_pool"], s["v_pool"], s["slots"], **s["kw"])
        return _state_of(s)
    if kind == "roundtrip":
        iva.kv_append(s["k"], s["v"], s["k_pool"], s["v_pool"], s["slots"])
        out = iva.kv_gather(s["k_pool"], s["v_pool"], s["tables"], s["lens"], out_len=s["out_len"])
        return [*out, *_state_of(s)]
    if kind == "gather":
        kw = dict(s["kw"], out_dtype=s["out_dtype"]) if s["kw"] else {}
        return iva.kv_gather(s["k_pool"], s["v_pool"], s["tables"], s["lens"], out_len=s["out_len"], **kw)
    if kind == "decode":
        if s["window"]:
            return [iva.paged_decode_attention(s["q"], s["k_pool"], s["v_pool"], s["tables"], s["lens"],
                                               window=s["window"], n_sink=s["sinks"], **s["kw"])]
        out = iva.paged_decode_append_attention(s["q"], s["k"], s["v"], s["k_pool"], s["v_pool"], s["tables"],
                                                s["lens"], **s["kw"])
        return [out, *_state_of(s)]
    return [iva.paged_prefill_attention(s["q"], s["k_pool"], s["v_pool"], s["tables"], s["lens"], s["start"],
                                        window=s["window"], n_sink=s["sinks"], max_query_len=s["longest"],
                                        **s["kw"])]


# ---------------------------------------------------------------- work, tolerance

def _row_bytes(c):
    """Bytes of one token's K and V (all kv heads) in the pages."""
    per = {"fp8": c["dim"] + 4, "fp32": 4 * c["dim"]}.get(c["pages"], 2 * c["dim"])
    return 2 * c["hkv"] * per


def _model_work(c, tokens, seqs):
    """(parameters read, flops) of one layer on `tokens` tokens, without attention."""
    d, kv = c["d_model"], c["d_model"] // c["heads"] * c["kv_heads"]
    weights = 2 * d * d + 2 * d * kv + 3 * 4 * d * d
    return weights, 2.0 * weights * tokens


def work(case):
    c, kind = case, case["kind"]
    if kind in ("block", "loop"):
        b, n, d = c["batch"], c["tokens"], c["d_model"]
        kv = d // c["heads"] * c["kv_heads"]
        weights, flops = _model_work(c, b * n, b)
        flops += 2.0 * b * n * (n + 1) * d
        if kind == "block":
            return {"bytes": 2.0 * weights + 4.0 * b * n * d, "flops": flops}
        t, layers, vocab = c["steps"], c["layers"], c["vocab"]
        per = 2.0 * (weights * layers + vocab * d)
        cached = sum(n + i + 1 for i in range(t))
        steps = 2.0 * b * t * (weights * layers + vocab * d) + 4.0 * b * cached * d * layers
        prompt = flops * layers + 2.0 * b * n * vocab * d
        return {"bytes": per * (1 + t) + 4.0 * b * layers * kv * (n + t + cached) + 2.0 * b * (n + t) * vocab,
                "flops": prompt + steps}
    lengths = _lengths(c)
    e = 4 if c["dtype"] == "fp32" else 2
    row = 2 * c["hkv"] * c["dim"] * e
    tables = 4.0 * sum(-(-n // BS) for n in lengths) + 4.0 * len(lengths)
    padded = float(len(lengths) * max(lengths) * row)
    if kind == "gather":
        return {"bytes": sum(lengths) * _row_bytes(c) + padded + tables, "flops": 0.0}
    if kind == "roundtrip":
        return {"bytes": 3.0 * sum(lengths) * row + padded + tables, "flops": 0.0}
    if kind == "decode":
        seen = [min(n, c["window"] + c["sinks"]) if c["window"] else n for n in lengths]
        q = 2.0 * len(lengths) * c["hq"] * c["dim"] * e
        return {"bytes": sum(seen) * _row_bytes(c) + q + tables + len(lengths) * row,
                "flops": 4.0 * c["hq"] * c["dim"] * sum(seen)}
    chunks = _chunks(c, lengths)
    if kind == "append":
        return {"bytes": sum(chunks) * (row + _row_bytes(c) + 4.0), "flops": 0.0}
    seen = [min(n, c["window"] + m + c["sinks"]) if c["window"] else n for n, m in zip(lengths, chunks)]
    return {"bytes": sum(seen) * _row_bytes(c) + 2.0 * sum(chunks) * c["hq"] * c["dim"] * e + tables,
            "flops": 4.0 * c["hq"] * c["dim"] * _pairs(c, lengths, chunks)}


def tolerance(case):
    c, kind = case, case["kind"]
    if kind in ("append", "roundtrip") or (kind == "gather" and c["pages"] != "fp8"):
        return "exact"  # rows are moved, or quantized by a stated rule: the same bits
    if kind == "block":
        return {"rel": 1e-2}
    if kind == "loop":
        return {"rel": 3e-2}
    # about four times the error against float64 that the attention kernels show
    return {"rel": {"fp32": 2e-6, "fp16": 1.2e-3, "bf16": 8e-3}[c["dtype"]]}


# ------------------------------------------------------------------------- exact

def _dequantized(c, x):
    """Rows as the pages hold them, in float64 (FP8: code / factor, factor 448 / max|row|)."""
    if c["pages"] != "fp8":
        return x.double()
    amax = x.float().abs().amax(dim=-1, keepdim=True)
    # (a tensor over a tensor: a number over a tensor multiplies by a rounded reciprocal)
    sf = torch.where(amax > 0, torch.full_like(amax, 448.0) / amax, torch.ones_like(amax))
    return (x.float() * sf).to(FP8).double() / sf.double()


def _attention(c, q, k, v, q_pos, k_pos):
    """q [n, Hq, D] at positions q_pos over k, v [m, Hkv, D] at k_pos, in float64."""
    n, hq, d = q.shape
    hkv = k.shape[1]
    g = hq // hkv
    qh = q.double().view(n, hkv, g, d).permute(1, 2, 0, 3).reshape(hkv, g * n, d)
    scores = torch.matmul(qh, k.permute(1, 2, 0).contiguous()) / math.sqrt(d)
    seen = k_pos[None, :] <= q_pos[:, None]
    if c.get("window"):
        seen &= (k_pos[None, :] > q_pos[:, None] - c["window"]) | (k_pos[None, :] < c["sinks"])
    scores.view(hkv, g, n, -1).masked_fill_(~seen, float("-inf"))
    out = torch.matmul(torch.softmax(scores, dim=-1), v.permute(1, 0, 2).contiguous())
    return out.view(hkv, g, n, d).permute(2, 0, 1, 3).reshape(n, hq, d)


def _norm(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def _block_exact(c, block, x):
    """One block in float64 on x [b, s, d]."""
    a, f = block.attention, block.ffn
    b, s, d = x.shape
    dim = d // c["heads"]
    pos = torch.arange(s, device=x.device)
    y = _norm(x, block.norm1.weight, 1e-6)
    q, k, v = (y @ p.weight.double().t() for p in (a.q_proj, a.k_proj, a.v_proj))
    o = torch.stack([_attention({}, q[i].view(s, -1, dim), k[i].view(s, -1, dim), v[i].view(s, -1, dim), pos, pos)
                     for i in range(b)])
    x = x + o.reshape(b, s, d) @ a.o_proj.weight.double().t()
    y = _norm(x, block.norm2.weight, 1e-6)
    up, gate = y @ f.up_proj.weight.double().t(), y @ f.gate_proj.weight.double().t()
    return x + (torch.nn.functional.silu(up) * gate) @ f.down_proj.weight.double().t()


@torch.no_grad()
def exact(case, seed):
    c, kind = case, case["kind"]
    if kind in ("append", "roundtrip"):
        return None
    if kind == "block":
        s = prepare(c, seed)
        return _block_exact(c, s["block"], s["x"].double())
    if kind == "loop":
        s = prepare(c, seed)
        m, ids = s["model"], torch.cat([s["prompt"], s["given"]], dim=1)
        x = m.token_embedding.weight.double()[ids] + m.position_embedding.weight.double()[:ids.shape[1]]
        for block in m.blocks:
            x = _block_exact(c, block, x)
        x = _norm(x[:, c["tokens"] - 1:], m.norm.weight, 1e-6)
        return x @ m.token_embedding.weight.double().t()
    lengths, keep, _, _ = _layout(c, seed)
    resident = [_resident(k, n).cuda() for k, n in zip(keep, lengths)]
    k, v = _rows(c, seed, sum(len(p) for p in resident))
    parts, at = [], 0
    for p in resident:
        parts.append((p, k[at:at + len(p)], v[at:at + len(p)]))
        at += len(p)
    if kind == "gather":
        out = [torch.zeros(len(lengths), c["hkv"], max(lengths), c["dim"], dtype=torch.float64, device="cuda")
               for _ in range(2)]
        for b, (p, kb, vb) in enumerate(parts):
            out[0][b, :, :len(p)] = _dequantized(c, kb).transpose(0, 1)
            out[1][b, :, :len(p)] = _dequantized(c, vb).transpose(0, 1)
        return out
    chunks = _chunks_of(c, lengths) if kind == "prefill" else [1] * len(lengths)
    q = _randn((sum(chunks), c["hq"], c["dim"]), seed, 4, DTYPES[c["dtype"]])
    outs, at = [], 0
    for n, m, (p, kb, vb) in zip(lengths, chunks, parts):
        outs.append(_attention(c, q[at:at + m], _dequantized(c, kb), _dequantized(c, vb),
                               torch.arange(n - m, n, device="cuda"), p))
        at += m
    out = torch.cat(outs)
    if kind == "decode" and not c["window"]:
        return [out] + [None] * (4 if c["pages"] == "fp8" else 2)
    return [out]
