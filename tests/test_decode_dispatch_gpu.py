"""Decode calls on both sides of every line of the launch choice (single launch against walk
+ merge by units and table width, two or four tiles per wave) against the same attention
evaluated as the stream walk's two halves, which take no such choice, or as append +
attention."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

# What two evaluations may differ by: the fp32 sums' order over <= 2000 keys of unit-variance
# values (2e-5), each side's rounding of the output (OUT, relative to it) and of every weight p
# to the products' operand type (WEIGHT, relative to the weighted mean of |v|; bf16 carries p
# as a pair).
OUT = {torch.float32: 0.0, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}
WEIGHT = {torch.float32: 0.0, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -16}




@pytest.mark.parametrize("batch,hkv,pages", [
    (1, 1, 1), (1, 8, 16), (1, 8, 17), (1, 8, 32), (1, 8, 33), (3, 5, 32), (31, 8, 8), (31, 8, 33),
    (32, 8, 64), (32, 8, 65), (127, 8, 3), (128, 8, 64), (130, 8, 65), (300, 7, 2),
    (1, 1, 100), (2, 8, 100), (4, 8, 50), (5, 5, 64), (4, 8, 101), (4, 8, 125)])
@pytest.mark.parametrize("dtype,d", [(torch.float16, 128), (torch.bfloat16, 64), (torch.float32, 64),
                                     (torch.bfloat16, 256), (torch.float16, 0)])
def test_decode_on_both_sides_of_the_launch_choice(iva, dev, batch, hkv, pages, dtype, d):
    fp8, d = d == 0, d or 128
    if fp8 and batch * pages > 9000:
        pytest.skip("covered by smaller batches")
    gen = torch.Generator(device=dev).manual_seed(batch * 1000 + pages)
    hq, n_pages = 2 * hkv, batch * pages + 1

    def randn(*shape):
        return torch.randn(shape, generator=gen, device=dev).to(dtype)

    table = torch.randperm(n_pages, generator=gen, device=dev)[:batch * pages].to(torch.int32).view(batch, pages)
    lens = torch.randint(1, 16 * pages + 1, (batch,), generator=gen, device=dev, dtype=torch.int32)
    lens[0] = 16 * pages
    if batch > 2:
        lens[1], lens[2] = 0, 1
        table[-1, pages // 2] = -1  # a page the sequence does not have
    ks, vs = iva.pool_shapes(n_pages, hkv, d, 16, iva.ops.FP8 if fp8 else dtype)
    rows = [randn(batch * pages * 16, hkv, d) for _ in range(2)]
    pool_dtype = iva.ops.FP8 if fp8 else dtype
    pools = [torch.zeros(s, dtype=pool_dtype, device=dev) for s in (ks, vs)]
    kw = {}
    if fp8:
        kw = {n: torch.ones(n_pages, hkv, 16, device=dev) for n in ("k_scale", "v_scale")}
    slots = (table.clamp(min=0).repeat_interleave(16, dim=1) * 16 + torch.arange(16, device=dev).repeat(pages)
             ).to(torch.int32).view(-1)
    iva.kv_append(rows[0], rows[1], *pools, slots, **kw)
    q, k_new, v_new = randn(batch, hq, d), randn(batch, hkv, d), randn(batch, hkv, d)

    def close(a, b, v_abs):
        a, b = a.double(), b.double()
        assert torch.isfinite(a).all()
        bound = 2e-5 + 2 * OUT[dtype] * b.abs() + 2 * WEIGHT[dtype] * 1.01 * v_abs
        assert ((a - b).abs() <= bound).all(), ((a - b).abs() - bound).max()

    def v_abs(k, v, k_scale=None, v_scale=None):
        """The weighted mean of |v| (FP8: of the codes' magnitudes over the factors)."""
        v = (v.view(torch.uint8) & 127).view(v.dtype) if fp8 else v.abs()
        kw = dict(k_scale=k_scale, v_scale=v_scale) if fp8 else {}
        return iva.paged_decode_attention(q, k, v, table, lens, **kw).double()

    got = iva.paged_decode_attention(q, *pools, table, lens, **kw)
    if not fp8:
        out = torch.empty_like(q)
        nbytes = iva.decode_workspace_bytes(batch, hq, hkv, d, 16, pages)
        ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
        iva.paged_decode_attention_partial(q, *pools, table, lens, out=out, workspace=ws)
        iva.paged_decode_attention_merge(q, *pools, table, lens, out=out, workspace=ws)
        close(got, out, v_abs(*pools))
    # the fused step on one copy of the pools, append then attention on another
    def clone(t):
        return t.view(torch.uint8).clone().view(t.dtype) if fp8 else t.clone()

    p1, p2 = [clone(t) for t in pools], [clone(t) for t in pools]
    k1, k2 = ({n: t.clone() for n, t in kw.items()} for _ in range(2))
    fused = iva.paged_decode_append_attention(q, k_new, v_new, *p1, table, lens, **k1)
    pos = (lens - 1).long()
    page = table.gather(1, (pos.clamp(min=0) // 16).view(-1, 1)).view(-1)
    new = torch.where((lens > 0) & (page >= 0), page * 16 + (pos % 16).int(), torch.full_like(lens, -1))
    iva.kv_append(k_new, v_new, *p2, new.to(torch.int32), **k2)
    close(fused, iva.paged_decode_attention(q, *p2, table, lens, **k2), v_abs(*p2, **k2))
    for a, b in zip(p1 + list(k1.values()), p2 + list(k2.values())):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
