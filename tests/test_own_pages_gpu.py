"""Attention without a cache runs on pages of its own that nobody has written before: whatever
their memory holds past the tokens has to stay unseen."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

# A row's projections, its attention and its output are rounded to the type about six times in
# a row on each side (2^-8, 2^-11); fp32: its sums of up to 512 products in another order.
REL = {torch.bfloat16: 6 * 2.0 ** -8, torch.float16: 6 * 2.0 ** -11, torch.float32: 2e-5}


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32], ids=str)
@pytest.mark.parametrize("window,sinks", [(None, 0), (20, 0), (20, 4)])
@pytest.mark.parametrize("heads,kv,dim", [(4, 4, 64), (4, 2, 128), (2, 1, 256)])
@pytest.mark.parametrize("tokens", [1, 17, 33, 47, 64])
def test_unwritten_memory_of_own_pages_is_not_seen(iva, dev, monkeypatch, tokens, heads, kv, dim, window, sinks,
                                                   dtype):
    M, made = iva.model, []

    class Dirty(M.OwnPages):
        def __init__(self, *args):
            super().__init__(*args)
            self._view.k_pool.fill_(float("nan"))
            self._view.v_pool.fill_(float("nan"))
            made.append(self)

    monkeypatch.setattr(M, "OwnPages", Dirty)
    cfg = dict(d_model=heads * dim, n_heads=heads, n_kv_heads=kv, n_layers=1, vocab_size=64, seq_len=64, dropout=0.0)
    torch.manual_seed(tokens)
    paged = M.PagedAttention(M.TransformerConfig(**cfg, attn_impl="hip_paged")).to(dev, dtype).eval()
    plain = M.AttentionTorch(M.TransformerConfig(**cfg)).to(dev, dtype).eval()
    plain.load_state_dict(paged.state_dict())
    x = torch.randn(3, tokens, heads * dim, device=dev).to(dtype)
    kw = dict(sliding_window=window, sink_cfg={"sink_tokens": sinks})
    padded = torch.ones(3, tokens, dtype=torch.long, device=dev)
    padded[0, : tokens // 3] = 0
    with torch.no_grad():
        for mask in ([None, padded] if tokens > 1 else [None]):
            got, ref = (m(x, attention_mask=mask, **kw)[0].double() for m in (paged, plain))
            if mask is not None:  # rows with no key left: the paged side gives zeros, as the plain one here
                assert torch.isfinite(ref).all()
            assert torch.isfinite(got).all()
            assert (got - ref).norm() <= REL[dtype] * ref.norm()
    assert len(made) == (2 if tokens > 1 else 1)
