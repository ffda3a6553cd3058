"""Where the layer kernels are taken.  The few-row linear kernel: by rows and widths, and not where its loss to the
library's products on the GPU outgrows what its fewer calls save the host.  The modules run on the meta device with the kernels stood
in, so that wide ones cost nothing.  RMSNorm's kernel: not for many very narrow rows."""
from __future__ import annotations

import pytest
import torch


@pytest.fixture
def taken(iva, monkeypatch):
    """The shapes [rows, k, columns...] of the calls that reach the kernel."""
    M, calls = iva.model, []

    def linear_rows(x, weights, norm=None, residual=None, swiglu_pair=False):
        k = x.shape[-1]
        calls.append([x.numel() // k, k] + [w.shape[0] for w in weights])
        outs = [x.new_empty((*x.shape[:-1], w.shape[0])) for w in weights[:1 if swiglu_pair else 3]]
        return outs if len(outs) > 1 else outs[0]

    def rms_norm(x, weight, eps, residual=None):
        return x if residual is None else (x, x)

    for name, value in dict(linear_rows=linear_rows, rms_norm=rms_norm, swiglu=lambda u, g: u,
                            _plain=lambda x: True, _plain_type=lambda x: True,
                            _plain_layout=lambda x: True, _plain_weight=lambda w, x: True).items():
        monkeypatch.setattr(M, name, value)
    # the attention itself: its projections' rows come out as they went in
    monkeypatch.setattr(M.PagedAttention, "_attend_rows",
                        lambda self, x, project, *a: (project(x)[0].reshape(x.shape), None))
    return calls


def _block(iva, d, hidden_mult=4, kv=None):
    cfg = iva.TransformerConfig(d_model=d, n_heads=d // 64, n_kv_heads=kv or d // 64, n_layers=1, vocab_size=64,
                                seq_len=8, dropout=0.0, hidden_mult=hidden_mult, attn_impl="hip_paged")
    with torch.device("meta"):
        return iva.model.TransformerBlock(cfg).eval()


def _x(rows, d):
    return torch.empty(rows, 1, d, device="meta")


@pytest.mark.parametrize("d,rows", [(64, 32), (1024, 1), (2048, 32), (4096, 32), (5120, 8), (8192, 8)])
def test_block_takes_the_kernel(iva, taken, d, rows):
    _block(iva, d)(_x(rows, d))
    assert taken == [[rows, d, d, d, d], [rows, d, d], [rows, d, 4 * d, 4 * d], [rows, 4 * d, d]]


@pytest.mark.parametrize("d,rows", [(1024, 33), (5120, 9), (8192, 16), (8192, 32)])
def test_wide_block_leaves_it(iva, taken, d, rows):
    _block(iva, d)(_x(rows, d))
    if rows > 16:  # at most the attention's projections alone take it there
        assert not taken
    else:
        assert taken == [[rows, d, d, d, d]]


@pytest.mark.parametrize("d,mult,rows,kernel", [
    (256, 4, 32, True), (1024, 8, 32, True), (2048, 4, 32, True), (3072, 4, 4, True), (8192, 4, 4, True),
    (3072, 4, 16, True), (4096, 4, 16, True), (2048, 8, 17, False), (3072, 4, 17, False), (4096, 4, 32, False),
    (8192, 4, 16, False), (1024, 4, 33, False)])
def test_ffn(iva, taken, d, mult, rows, kernel):
    _block(iva, d, mult).ffn(_x(rows, d))
    assert bool(taken) == kernel


@pytest.mark.parametrize("d,rows,qkv,o", [
    (1024, 32, True, True), (2048, 32, True, True), (3072, 16, True, True), (4096, 17, True, False),
    (5120, 1, True, False), (8192, 16, True, False), (8192, 17, False, False), (64, 33, False, False)])
def test_attention_alone(iva, taken, d, rows, qkv, o):
    _block(iva, d).attention(_x(rows, d))
    assert taken == [[rows, d, d, d, d]] * qkv + [[rows, d, d]] * o


@pytest.mark.parametrize("d,vocab,rows,kernel", [
    (1024, 32000, 16, True), (256, 32000, 1, True), (2048, 4096, 16, True), (4096, 512, 16, True), (512, 512, 17, False),
    (768, 50304, 1, False), (1024, 65536, 4, False), (1536, 32000, 1, False), (2048, 32000, 1, False),
    (4096, 32000, 8, False), (8192, 512, 1, False), (8192, 128256, 16, False)])
def test_head(iva, taken, d, vocab, rows, kernel):
    head = iva.Transformer.__new__(iva.Transformer)
    torch.nn.Module.__init__(head)
    with torch.device("meta"):
        head.token_embedding, head.lm_head = torch.nn.Embedding(vocab, d), None
    assert head.logits(_x(rows, d)).shape == (rows, 1, vocab)
    assert taken == [[rows, d, vocab]] * kernel


@pytest.mark.parametrize("d,rows,kernel", [
    (8, 1 << 16, True), (8, (1 << 16) + 1, False), (24, 1 << 16, True), (24, 1 << 20, False),
    (32, 1 << 20, True), (4096, 1 << 20, True)])
def test_norm_of_many_narrow_rows_leaves_the_kernel(iva, taken, monkeypatch, d, rows, kernel):
    M, norms = iva.model, []
    monkeypatch.setattr(M, "rms_norm", lambda x, w, eps: norms.append(tuple(x.shape)) or x)
    cfg = iva.TransformerConfig(d_model=d, n_heads=1, n_kv_heads=1, n_layers=1, vocab_size=64, seq_len=8, dropout=0.0)
    with torch.device("meta"):
        norm = M.RMSNorm(cfg)
    norm(_x(rows, d))
    assert bool(norms) == kernel
