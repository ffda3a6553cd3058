"""Decoder-layer kernels (RMSNorm, SwiGLU, few-row linear layers) against float64, and the
block that fuses them against the same block run module by module.

Bounds: with u = 2^-8 (bf16, 8 significant bits) / 2^-11 (fp16, 11) the largest relative
error of rounding one value to nearest, an output
is off by at most u |y| for its own rounding plus what its operands' roundings and the fp32
sums (k terms, 2^-24 each) carry into it; each test states that sum.
"""
from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

U = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}
DTYPES = [torch.bfloat16, torch.float16]


def _randn(shape, seed, dev, dtype, scale=1.0):
    gen = torch.Generator(device=dev).manual_seed(seed)
    return (torch.randn(shape, generator=gen, device=dev) * scale).to(dtype)


def _norm64(x, w, eps=1e-6):
    x = x.double()
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)
    return y if w is None else y * w.double()


def _within(got, ref, bound):
    worst = ((got.double() - ref).abs() - bound).max().item()
    assert worst <= 0, f"over the bound by {worst}"


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows,d", [(1, 8), (3, 512), (5, 520), (16, 1024), (9, 2056), (4, 8192)])
def test_rms_norm(iva, dev, dtype, rows, d):
    ops = iva.ops
    x, r, w = (_randn(s, i, dev, dtype) for i, s in enumerate([(rows, d), (rows, d), (d,)]))
    # two roundings (y, then y * w) and the fp32 root: 3 u |y|; among fp16's subnormals
    # (spacing 2^-24) a rounding is off by up to 2^-25 instead, the first one times |w| < 8
    tiny = 9 * 2.0 ** -25
    _within(ops.rms_norm(x, w, 1e-6), _norm64(x, w), 3 * U[dtype] * _norm64(x, w).abs() + tiny)
    _within(ops.rms_norm(x, None, 1e-6), _norm64(x, None), 2 * U[dtype] * _norm64(x, None).abs() + tiny)
    total, y = ops.rms_norm(x, w, 1e-6, residual=r)
    assert torch.equal(total, x + r)
    ref = _norm64(x + r, w)
    _within(y, ref, 3 * U[dtype] * ref.abs() + tiny)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n", [8, 2048, 4096 + 8, 100008])
def test_swiglu(iva, dev, dtype, n):
    up, gate = _randn(n, 1, dev, dtype, 4.0), _randn(n, 2, dev, dtype)
    up[:6] = torch.tensor([0.0, -0.0, 300.0, -300.0, float("inf"), float("nan")], dtype=dtype)
    got, ref = iva.ops.swiglu(up, gate), F.silu(up.double()) * gate.double()
    assert torch.equal(got[4:6].isnan(), ref[4:6].isnan())
    ok = ref.isfinite()
    # one rounding, and exp / reciprocal at 2^-21; 2^-24 absolute covers fp16's subnormals
    _within(got[ok], ref[ok], 1.01 * U[dtype] * ref[ok].abs() + 2.0 ** -24)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("k,n", [(64, 16), (320, 48), (1024, 32), (1088, 16), (2048, 64), (4160, 32)])
@pytest.mark.parametrize("m", [1, 4, 5, 16, 17, 32])
def test_linear_rows(iva, dev, dtype, m, k, n):
    ops = iva.ops
    x = _randn((m, k), 3, dev, dtype)
    w = [_randn((n * (i + 1), k), 4 + i, dev, dtype, k ** -0.5) for i in range(3)]
    res, up = _randn((m, n), 8, dev, dtype), _randn((n, k), 9, dev, dtype, k ** -0.5)
    sums = 2.0 ** -23 * k ** 0.5 * 4  # the fp32 sums of k products of unit variance / k

    def check(got, ref, extra=0.0):
        _within(got, ref, 1.01 * U[dtype] * ref.abs() + sums + extra)

    for got, wi in zip(ops.linear_rows(x, w), w):
        check(got, x.double() @ wi.double().t())
    check(ops.linear_rows(x, w[:1], residual=res), x.double() @ w[0].double().t() + res.double())
    ug = x.double() @ up.double().t(), x.double() @ w[0].double().t()
    check(ops.linear_rows(x, [w[0], up], swiglu_pair=True), F.silu(ug[0]) * ug[1],
          2 * sums * (1 + ug[0].abs() + ug[1].abs()))
    if m <= ops.LINEAR_NORM_MAX_ROWS and k <= ops.LINEAR_NORM_MAX_K:
        nw = _randn(k, 10, dev, dtype)
        y = ops.rms_norm(x, nw, 1e-6)
        fused = ops.linear_rows(x, w, norm=(nw, 1e-6))
        pair = ops.linear_rows(x, [w[0], up], norm=(nw, 1e-6), swiglu_pair=True)
        if dtype == torch.float16 or m <= 4:  # normalized as the kernel alone does
            for got, alone in zip(fused, ops.linear_rows(y, w)):
                assert torch.equal(got, alone)
            assert torch.equal(pair, ops.linear_rows(y, [w[0], up], swiglu_pair=True))
        else:  # x * nw rounded once (u each product), the sums scaled by 1 / rms
            yd = _norm64(x, nw)
            for got, wi in zip(fused, w):
                check(got, yd @ wi.double().t(), 1.01 * U[dtype] * (yd.abs() @ wi.double().abs().t()))
            e = [1.01 * U[dtype] * (yd.abs() @ t.double().abs().t()) for t in (up, w[0])]
            u, g = yd @ up.double().t(), yd @ w[0].double().t()
            # |d silu| <= 1.1 |du|
            check(pair, F.silu(u) * g, 1.2 * e[0] * (g.abs() + e[1]) + F.silu(u).abs() * e[1]
                  + 2 * sums * (1 + u.abs() + g.abs()))


def test_linear_rows_many_tiles(iva, dev):
    """More column tiles than workgroups: each takes several, an odd number of them."""
    n, k = 16 * (2 * 1024 + 333), 1024
    x, w = _randn((16, k), 1, dev, torch.bfloat16), _randn((n, k), 2, dev, torch.bfloat16, k ** -0.5)
    ref = x.double() @ w.double().t()
    _within(iva.ops.linear_rows(x, (w,)), ref, 1.01 * U[torch.bfloat16] * ref.abs() + 2.0 ** -16)


@pytest.mark.parametrize("d_model,heads,kv", [(256, 4, 2), (1024, 16, 16), (2560, 10, 10)])
@pytest.mark.parametrize("batch,tokens", [(1, 2), (16, 1), (2, 12), (3, 40)])
def test_fused_block_matches_modules(iva, dev, d_model, heads, kv, batch, tokens):
    """The fused block and the same block with a hook on a submodule, which makes it run
    module by module (and the hook fire)."""
    M = iva.model
    cfg = M.TransformerConfig(d_model=d_model, n_heads=heads, n_kv_heads=kv, n_layers=1, vocab_size=64,
                              seq_len=128, dropout=0.1, attn_impl="hip_paged")
    torch.manual_seed(5)
    block = M.Transformer(cfg).to(dev, torch.bfloat16).eval().blocks[0]
    x = _randn((batch, tokens, d_model), 6, dev, torch.bfloat16)
    with torch.no_grad():
        fused = block(x)[0]
        calls = []
        hooks = [m.register_forward_hook(lambda mod, i, o: calls.append(type(mod).__name__))
                 for m in (block.attention.o_proj, block.ffn.down_proj, block.norm2)]
        alone = block(x)[0]
        for h in hooks:
            h.remove()
        with torch.enable_grad():
            grad = block.norm1(x.requires_grad_())
        assert grad.requires_grad
    assert sorted(calls) == ["Linear", "Linear", "RMSNorm"]
    # both round every intermediate once or twice to bf16, six in a row
    err = (fused.double() - alone.double()).norm() / alone.double().norm()
    assert err <= 6 * U[torch.bfloat16], err


@pytest.mark.parametrize("kw", [{}, dict(kv_cache_dtype="fp8"), dict(sliding_window=48, sink_tokens=4),
                                dict(n_kv_heads=1)])
@pytest.mark.parametrize("batch", [1, 16, 19])
def test_decode_step_in_one_call_matches_modules(iva, dev, batch, kw):
    """Decode steps whose blocks are one call each, and the same steps module by module (a
    hook on a submodule of every block), from the same cached prompt across a page boundary."""
    M = iva.model
    cfg = M.TransformerConfig(d_model=512, n_heads=8, **{"n_kv_heads": 2, **kw}, n_layers=3, vocab_size=64,
                              seq_len=256, dropout=0.1, attn_impl="hip_paged")
    torch.manual_seed(7)
    model = M.Transformer(cfg).to(dev, torch.bfloat16).eval()
    ids = torch.randint(0, 64, (batch, 61 + 5), device=dev, generator=torch.Generator(dev).manual_seed(1))

    def steps():
        cache = model.new_kv_cache(batch, 66)
        out = [model(ids[:, :61], kv_cache=cache)["logits"][:, -1]]
        for t in range(61, 66):
            out.append(model(ids[:, t:t + 1], kv_cache=cache)["logits"][:, -1])
        kv = [cache.layer_kv(i) for i in range(3)]
        n = cache.seq_len
        cache.free()
        return torch.stack(out), kv, n

    with torch.no_grad():
        fused, kv, n = steps()
        calls = []
        hooks = [b.ffn.up_proj.register_forward_hook(lambda m, i, o: calls.append(1)) for b in model.blocks]
        alone, kv2, n2 = steps()
        for h in hooks:
            h.remove()
    assert len(calls) == 3 * 6 and n == n2 == 66
    # three blocks of about six bf16 roundings in a row (FP8 codes flip at their 2^-4 steps)
    tol = 18 * U[torch.bfloat16] * (4 if cfg.kv_cache_dtype else 1)
    for a, b in [(fused, alone)] + [(x, y) for p, q in zip(kv, kv2) for x, y in zip(p, q)]:
        assert (a.double() - b.double()).norm() <= tol * b.double().norm()


@pytest.mark.parametrize("window,sinks", [(48.0, 4), (48.9, 4), (0.0, 4), (None, 0)])
def test_decode_step_window_types(iva, dev, window, sinks):
    """A window read from a configuration as a float is truncated, as the attention ops do."""
    M = iva.model
    cfg = M.TransformerConfig(d_model=256, n_heads=4, n_layers=1, vocab_size=64, seq_len=128, dropout=0.0,
                              attn_impl="hip_paged")
    torch.manual_seed(3)
    block = M.Transformer(cfg).to(dev, torch.bfloat16).eval().blocks[0]
    prompt, x = (_randn((2, n, 256), n, dev, torch.bfloat16) for n in (80, 1))

    def step(w):
        cache = iva.PagedKVCache(2, 4, 64, 0, dev, torch.bfloat16, num_layers=1, max_seq_len=96)
        kw = dict(sliding_window=w, sink_cfg={"sink_tokens": sinks})
        with torch.no_grad():
            return torch.stack([block(prompt, kv_cache=cache, **kw)[0][:, -1:], block(x, kv_cache=cache, **kw)[0]])

    assert torch.equal(step(window), step(None if window is None else int(window)))


@pytest.mark.parametrize("lengths,n", [([16, 16], 16), ([40, 40, 40], 1), ([33, 5, 100], 7), ([3], 5)])
def test_chunk_slots_match_the_pool(iva, dev, lengths, n):
    """Slots found on the device equal the allocator's; positions without a page give -1."""
    pool = iva.PagedKVPool(64, 1, 64, num_layers=1, dtype=torch.float16, device=dev, max_seqs=8)
    want = []
    for i, length in enumerate(lengths):
        pool.add_sequence(i)
        pool.allocate(i, length)
        first = max(length - n, 0)
        want += [-1] * (n - (length - first)) + pool.slots(i, range(first, length)).tolist()
    bt, ctx = pool.device_tables(range(len(lengths)))
    assert iva.ops.chunk_slots(bt, ctx, n).tolist() == want
    assert iva.ops.chunk_slots(bt[:, :1].contiguous(), ctx, 1).tolist() == [
        pool.slots(i, [length - 1])[0] if length <= 16 else -1 for i, length in enumerate(lengths)]
    assert iva.ops.chunk_slots(bt, ctx, 0).numel() == 0
