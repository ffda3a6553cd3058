"""The decoder layer's modules under torch's transforms: whatever mode the layer kernels do
not take, the torch operators run (CPU; ``is_cuda`` is stood in where a GPU tensor is meant)."""
from __future__ import annotations

import pytest
import torch


def _model(iva, dtype=torch.float32):
    cfg = iva.TransformerConfig(d_model=64, n_heads=2, n_layers=1, vocab_size=64, seq_len=32, dropout=0.0,
                                attn_impl="torch")
    torch.manual_seed(0)
    return iva.Transformer(cfg).to(dtype).eval()


def _module(model, name):
    block = model.blocks[0]
    return {"norm": block.norm1, "ffn": block.ffn, "block": lambda x: block(x)[0]}[name]


TRANSFORMS = {
    "vmap": lambda f, x: torch.func.vmap(f)(x[None]),
    "grad": lambda f, x: torch.func.grad(lambda t: f(t).float().sum())(x),
    "jvp": lambda f, x: torch.func.jvp(f, (x,), (torch.ones_like(x),))[1],
}


@pytest.mark.parametrize("transform", TRANSFORMS)
@pytest.mark.parametrize("name", ["norm", "ffn", "block"])
@pytest.mark.parametrize("grad", [False, True])
def test_functorch_transforms_of_16bit_gpu_tensors(iva, monkeypatch, name, transform, grad):
    f = _module(_model(iva, torch.bfloat16), name)
    x = torch.randn(2, 3, 64, dtype=torch.bfloat16)
    with torch.set_grad_enabled(grad):
        ref = TRANSFORMS[transform](f, x)
        monkeypatch.setattr(torch.Tensor, "is_cuda", True)
        got = TRANSFORMS[transform](f, x)
        monkeypatch.undo()
    assert torch.equal(got, ref)


def _compiled(model, name, x, grad):
    f = _module(model, name) if name != "model" else lambda ids: model(ids)["logits"]
    with torch.set_grad_enabled(grad):
        torch._dynamo.reset()
        return torch.compile(f, backend="eager", fullgraph=True)(x), f(x)


@pytest.mark.parametrize("name", ["norm", "ffn", "block", "model"])
@pytest.mark.parametrize("grad", [False, True])
def test_compiles_in_one_graph(iva, name, grad):
    x = torch.randint(0, 64, (2, 4)) if name == "model" else torch.randn(2, 4, 64)
    got, ref = _compiled(_model(iva), name, x, grad)
    assert torch.equal(got, ref)


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["norm", "ffn", "block", "model"])
@pytest.mark.parametrize("grad", [False, True])
def test_compiles_in_one_graph_16bit(iva, dev, name, grad):
    """The graph holds the torch operators; without grad the plain call runs the layer kernels."""
    model = _model(iva, torch.bfloat16).to(dev)
    x = (torch.randint(0, 64, (2, 4), device=dev) if name == "model"
         else torch.randn(2, 4, 64, device=dev, dtype=torch.bfloat16))
    got, ref = _compiled(model, name, x, grad)
    # (norm: the torch operators round twice, as the kernel; a block rounds six times in a row)
    assert (got - ref).float().norm() <= 6 * 2.0 ** -8 * ref.float().norm()


@pytest.mark.parametrize("affine", [False, True])
def test_norm_scripts(iva, affine):
    cfg = iva.TransformerConfig(d_model=64, n_heads=2, n_layers=1, vocab_size=64, elementwise_affine=affine)
    norm, x = iva.model.RMSNorm(cfg), torch.randn(3, 64)
    with torch.no_grad():
        assert torch.equal(torch.jit.script(norm)(x), norm(x))
