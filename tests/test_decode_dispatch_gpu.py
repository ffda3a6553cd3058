"""Decode calls on both sides of every line of the launch choice (single launch against walk
+ merge by units and table width, two or four tiles per wave) against float64 attention over
the rows that the pools hold."""
from __future__ import annotations

import random

import pytest
import torch

# What an output may be off by: the fp32 sums over <= 3200 keys of unit-variance values (2e-5),
# the rounding of the output (OUT, relative to it) and of every weight p to the products'
# operand type (WEIGHT, relative to the weighted mean of |v|; bf16 carries p as a pair).
OUT = {torch.float32: 0.0, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}
WEIGHT = {torch.float32: 0.0, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -16}

SHAPES = [  # batch, kv heads, table width
    (1, 1, 1), (1, 8, 16), (1, 8, 17), (1, 8, 32), (1, 8, 33), (3, 5, 32), (31, 8, 8), (31, 8, 33),
    (32, 8, 64), (32, 8, 65), (127, 8, 3), (128, 8, 64), (130, 8, 65), (300, 7, 2),
    (1, 1, 100), (2, 8, 100), (4, 8, 50), (5, 5, 64), (4, 8, 101), (4, 8, 125), (7, 8, 100), (6, 8, 120),
    (16, 8, 125), (1, 1, 200), (2, 8, 200),
    (150, 8, 3), (150, 8, 8), (520, 8, 2), (520, 8, 5)]  # four or more units per CU


def _lens(batch, pages):
    r = random.Random(batch * 1000 + pages)
    lens = [r.randint(1, 16 * pages) for _ in range(batch)]
    lens[0] = 16 * pages
    if batch > 2:
        lens[1], lens[2] = 0, 1
    return lens


def test_shapes_cover_the_walks_tile_counts():
    """Tables too wide for a single launch at any type (16-bit pages to D 128): two tiles per wave
    up to 1600 tiles and 192 per unit; then 800 waves up to 60 tiles per unit; else four tiles."""
    tiles = [(sum(-(-n // 16) for n in _lens(b, pages)) * hkv, b * hkv) for b, hkv, pages in SHAPES
             if pages > (64 if b * hkv >= 256 else 32)]
    assert sum(t <= min(1600, 192 * u) for t, u in tiles) >= 3
    assert sum(192 * u < t <= 1600 for t, u in tiles) >= 1
    assert sum(1600 < t < min(3200, 60 * u) for t, u in tiles) >= 1
    assert sum(1600 < t <= 3200 and t > 60 * u for t, u in tiles) >= 1
    assert sum(t > 3200 for t, u in tiles) >= 2


def _rows(k_pool, v_pool, k_scale=None, v_scale=None):
    """K and V of every page in float64, [page, row, kv head, dim]."""
    p, h, nch, bs, x = k_pool.shape
    d = nch * x
    k = k_pool.double().permute(0, 3, 1, 2, 4).reshape(p, bs, h, d)
    if k_scale is None:
        return k, v_pool.double().permute(0, 3, 1, 2)
    # FP8: V's bytes lie in order [dim % 16][row / 4][dim / 16][row % 4]; value = code / factor
    v = v_pool.double().reshape(p, h, 16, 4, d // 16, 4).permute(0, 3, 5, 1, 4, 2).reshape(p, bs, h, d)
    return k / k_scale.double().transpose(1, 2)[..., None], v / v_scale.double().transpose(1, 2)[..., None]


def _attention64(q, rows, table, lens):
    """Attention of each sequence's query over its first lens keys, those on pages it does not
    have left out, and the weighted mean of |v|; both float64."""
    k, v = rows
    out, v_abs = torch.zeros(q.shape, dtype=torch.float64, device=q.device), torch.zeros(
        q.shape, dtype=torch.float64, device=q.device)
    h, d = k.shape[2:]
    for b, n in enumerate(lens):
        at = [t * 16 + r for t in range(-(-n // 16)) if int(table[b, t]) >= 0 for r in range(min(16, n - 16 * t))]
        if not at:
            continue
        pages = table[b].to(q.device).long()
        pos = torch.tensor(at, device=q.device)
        kb, vb = (t[pages[pos // 16], pos % 16].permute(1, 0, 2).contiguous() for t in (k, v))  # [h, n, d]
        qb = q[b].double().view(h, -1, d)
        w = torch.softmax(torch.matmul(qb, kb.transpose(1, 2).contiguous()) * d ** -0.5, dim=-1)
        out[b] = torch.matmul(w, vb).view(-1, d)
        v_abs[b] = torch.matmul(w, vb.abs()).view(-1, d)
    return out, v_abs


@pytest.mark.gpu
@pytest.mark.parametrize("batch,hkv,pages", SHAPES)
@pytest.mark.parametrize("dtype,d", [(torch.float16, 128), (torch.bfloat16, 64), (torch.float32, 64),
                                     (torch.bfloat16, 256), (torch.float16, 0), (torch.bfloat16, 0)])
def test_decode_on_both_sides_of_the_launch_choice(iva, dev, batch, hkv, pages, dtype, d):
    fp8, d = d == 0, d or 128
    gen = torch.Generator(device=dev).manual_seed(batch * 1000 + pages)
    hq, n_pages = 2 * hkv, batch * pages + 1

    def randn(*shape):
        return torch.randn(shape, generator=gen, device=dev).to(dtype)

    order = torch.randperm(n_pages, generator=torch.Generator().manual_seed(batch + pages))
    host_table = order[:batch * pages].to(torch.int32).view(batch, pages).clone()
    n_keys = _lens(batch, pages)
    slots = (host_table.repeat_interleave(16, dim=1) * 16 + torch.arange(16).repeat(pages)).to(torch.int32).view(-1)
    if batch > 2:
        host_table[-1, pages // 2] = -1  # a page the sequence does not have
    table, lens = host_table.to(dev), torch.tensor(n_keys, dtype=torch.int32, device=dev)
    pool_dtype = iva.ops.FP8 if fp8 else dtype
    pools = [torch.zeros(s, dtype=pool_dtype, device=dev) for s in iva.pool_shapes(n_pages, hkv, d, 16, pool_dtype)]
    kw = {}
    if fp8:
        kw = {n: torch.ones(n_pages, hkv, 16, device=dev) for n in ("k_scale", "v_scale")}
    iva.kv_append(randn(batch * pages * 16, hkv, d), randn(batch * pages * 16, hkv, d), *pools, slots.to(dev), **kw)
    q, k_new, v_new = randn(batch, hq, d), randn(batch, hkv, d), randn(batch, hkv, d)

    def close(got, exact):
        ref, v_abs = exact
        got = got.double()
        assert torch.isfinite(got).all()
        bound = 2e-5 + OUT[dtype] * ref.abs() + WEIGHT[dtype] * 1.01 * v_abs
        assert ((got - ref).abs() <= bound).all(), ((got - ref).abs() - bound).max()

    exact = _attention64(q, _rows(*pools, **kw), host_table, n_keys)
    close(iva.paged_decode_attention(q, *pools, table, lens, **kw), exact)
    if not fp8:  # the stream walk's two halves
        out = torch.empty_like(q)
        nbytes = iva.decode_workspace_bytes(batch, hq, hkv, d, 16, pages)
        ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
        iva.paged_decode_attention_partial(q, *pools, table, lens, out=out, workspace=ws)
        iva.paged_decode_attention_merge(q, *pools, table, lens, out=out, workspace=ws)
        close(out, exact)
    # the fused step on one copy of the pools, the append on another

    def clone(t):
        return t.view(torch.uint8).clone().view(t.dtype) if fp8 else t.clone()

    p1, p2 = [clone(t) for t in pools], [clone(t) for t in pools]
    k1, k2 = ({n: t.clone() for n, t in kw.items()} for _ in range(2))
    fused = iva.paged_decode_append_attention(q, k_new, v_new, *p1, table, lens, **k1)
    pos = (lens - 1).long()
    page = table.gather(1, (pos.clamp(min=0) // 16).view(-1, 1)).view(-1)
    new = torch.where((lens > 0) & (page >= 0), page * 16 + (pos % 16).int(), torch.full_like(lens, -1))
    iva.kv_append(k_new, v_new, *p2, new.to(torch.int32), **k2)
    close(fused, _attention64(q, _rows(*p2, **k2), host_table, n_keys))
    for a, b in zip(p1 + list(k1.values()), p2 + list(k2.values())):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
