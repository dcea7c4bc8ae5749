"""An op whose main input is a module's parameter (the relative table's
LayerNorm) runs its implementation directly: the same kernel, so equal to the
custom op to the last bit, in the output and in every gradient; a graph of the
gradient still ends in the op's own error."""

from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("amp", [False, True], ids=["fp32", "autocast"])
def test_parameter_runs_directly(amp, gpu):
    from deberta_amd import RelativeEmbeddings
    from deberta_amd import blocks  # noqa: F401

    torch.manual_seed(0)
    cfg = SimpleNamespace(hidden_size=192, position_buckets=24, max_relative_positions=64, layer_norm_eps=1e-7)
    rel = RelativeEmbeddings(cfg).to(gpu)
    w, ln = rel.rel_embeddings.weight, rel.LayerNorm
    leaves = [w, ln.weight, ln.bias]
    with torch.autocast("cuda", dtype=torch.bfloat16, enabled=amp):
        y = rel()
        want = torch.ops.deberta_amd.add_ln(w, None, None, ln.weight, ln.bias, float(ln.eps), torch.float32)[0]
    assert "AddLnFunction" in type(y.grad_fn).__name__
    assert torch.equal(y, want)
    dy = torch.randn_like(y)
    for a, b in zip(torch.autograd.grad(y, leaves, dy), torch.autograd.grad(want, leaves, dy)):
        assert torch.equal(a, b)
    y = rel()
    (g,) = torch.autograd.grad((y * y).sum(), w, create_graph=True)
    with pytest.raises(RuntimeError):
        torch.autograd.grad(g.sum(), w)
