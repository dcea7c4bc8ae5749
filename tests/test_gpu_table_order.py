"""Table gradients in the tables' memory order: [2A, H, D] projections seen as
[H, 2A, D] against the same values contiguous (the fold sums in a fixed order
but its accumulators take atomic adds, so equal to their rounding: 2^-20 of
scale in fp32, one bf16 step), and a projection's gradient without a copy."""

from __future__ import annotations

import pytest
import torch

from tests._cases import Case, make_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize(
    "H,L,D,types,buckets",
    [(1, 33, 64, "c2p|p2c", 16), (3, 130, 32, "c2p", 16), (2, 257, 64, "p2c", 24), (4, 600, 64, "c2p|p2c", 32)],
)
def test_gradient_order(H, L, D, types, buckets, dtype, gpu):
    from deberta_amd import disentangled_attention

    c = Case(B=2, H=H, L=L, D=D, types=types, buckets=buckets, max_pos=2 * buckets, seed=H)
    x = make_inputs(c)
    dev = lambda t: t.to(gpu, dtype)
    got = []
    for rows_first in (False, True):
        q, k, v = (dev(x[n]).requires_grad_() for n in ("q", "k", "v"))
        tabs, leaves = [], []
        for n, name in (("kr", "c2p"), ("qr", "p2c")):
            if name not in types:
                tabs.append(None)
                continue
            t = dev(x[n])
            leaf = (t.permute(1, 0, 2).contiguous() if rows_first else t).detach().requires_grad_()
            leaves.append(leaf)
            tabs.append(leaf.permute(1, 0, 2) if rows_first else leaf)
        out = disentangled_attention(
            q, k, v, *tabs, None, None, position_buckets=c.buckets, max_relative_positions=c.max_pos, att_type=types,
            layout="blhd",
        )
        grads = torch.autograd.grad(out, [q, k, v, *leaves], dev(x["dout"]))
        assert all(g.is_contiguous() for g in grads)
        got.append([out, *grads[:3]] + [g.permute(1, 0, 2) if rows_first else g for g in grads[3:]])
    for a, b in zip(*got):
        a, b = a.float(), b.float()
        tol = (2.0**-20 if dtype == torch.float32 else 2.0**-7) * float(a.abs().max())
        assert float((a - b).abs().max()) <= tol
