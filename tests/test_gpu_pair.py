"""Dense pair masks as bits and tile flags (dsa_pair.h) where the pass and the
tile lists can go wrong: ends of 64-key tiles and 128-key blocks, masks
broadcast over the batch or given per head, tiles without a kept pair, tiles
kept whole, rows without a live query, dropout beside the mask, the p2p query
rows and far blocks.  The op against the CPU oracle (the parity suite's
bounds: fp32 1e-4 of scale, bf16 2e-2), and the forward with its workspace
(bits) against the forward without one (bytes)."""

from __future__ import annotations

import ctypes
import math

import pytest
import torch

from tests._cases import Case, hip_run, make_inputs, max_abs, max_rel, oracle_run

pytestmark = pytest.mark.gpu


def _window(B, L, w, heads=1):
    i = torch.arange(L)
    keep = ((i[:, None] - i[None, :]).abs() <= w)[None, None].repeat(B, heads, 1, 1)
    for h in range(heads):
        keep[:, h, 3 * h :: 17, h] = True  # another pattern per head
    return keep


def _mask(kind: str, B: int, L: int, H: int, g: torch.Generator) -> torch.Tensor:
    if kind == "window":
        return _window(B, L, 9)
    if kind == "heads":
        return _window(B, L, 40, H)
    if kind == "broadcast":
        return _window(1, L, 70)
    if kind == "causal":
        return torch.ones(L, L, dtype=torch.bool).tril()[None, None].repeat(B, 1, 1, 1)
    if kind == "empty":  # row 0 keeps nothing, the last query only itself
        keep = torch.zeros(B, 1, L, L, dtype=torch.bool)
        keep[-1, 0, -1, -1] = True
        return keep
    keep = torch.rand(B, 1, L, L, generator=g) < 0.02
    keep[0, 0, : L // 2] = True  # whole tiles kept
    keep[:, 0, L // 3] = False   # a dead row
    return keep


_CASES = [
    ("window", Case(B=2, H=2, L=128, D=64, seed=1)),
    ("window", Case(B=1, H=3, L=193, D=32, seed=2)),
    ("heads", Case(B=2, H=3, L=130, D=64, seed=3)),
    ("broadcast", Case(B=3, H=2, L=257, D=64, types="c2p", seed=4)),
    ("causal", Case(B=2, H=2, L=300, D=64, dropout=0.1, seed=5)),
    ("causal", Case(B=1, H=1, L=1, D=64, seed=6)),
    ("empty", Case(B=2, H=1, L=140, D=64, seed=7)),
    ("mixed", Case(B=2, H=2, L=320, D=64, types="p2c", seed=8)),
    ("mixed", Case(B=2, H=2, L=450, D=32, types="c2p|p2c|p2p", dropout=0.1, seed=9)),
    ("window", Case(B=1, H=2, L=600, D=64, buckets=32, max_pos=64, seed=10)),  # far blocks, none of them kept
    ("mixed", Case(B=1, H=2, L=600, D=64, buckets=32, max_pos=64, dropout=0.1, seed=11)),
]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("kind,c", _CASES, ids=[f"{k}-{c.seed}" for k, c in _CASES])
def test_pair_mask_forms(kind, c, dtype, gpu):
    x = make_inputs(c)
    x["mask"] = _mask(kind, c.B, c.L, c.H, torch.Generator().manual_seed(c.seed))
    ref = oracle_run(c, x, dtype)
    from deberta_amd import masks

    kernel_masks = masks.kernel_masks
    try:  # the mask as given, per head too
        masks.kernel_masks = lambda m, B, Lq, Lk, dev, **kw: kernel_masks(
            m, B, Lq, Lk, dev, segments_from_dense=False, heads=c.H
        )
        got = hip_run(c, x, dtype, gpu)
    finally:
        masks.kernel_masks = kernel_masks
    for name, r in ref.items():
        assert torch.isfinite(got[name]).all(), name
        scale = float(r.abs().max()) if r.numel() else 0.0
        if dtype == torch.float32:
            err, tol = (max_rel(got[name], r), 1e-4) if scale > 1e-6 else (max_abs(got[name], r), 1e-6)
        else:  # table gradients sum many pairs: held to their scale
            err, tol = (max_rel(got[name], r) if scale > 1.0 else max_abs(got[name], r)), 2e-2
        assert err <= tol, (kind, c, name, err)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("L", [96, 257])
def test_forward_without_workspace_equals_bits(L, dtype, gpu):
    """The same products in the same order: equal to the last bit (no far
    blocks at these lengths)."""
    from deberta_amd import _lib, ops
    from deberta_amd.masks import kernel_masks
    from deberta_amd.relpos import relative_offset_table

    lib = _lib.load()
    B, H, D, A = 2, 2, 64, 256
    g = torch.Generator().manual_seed(L)
    mk = lambda *s: torch.randn(*s, generator=g).to(gpu, dtype)
    q, k, v, kr, qr = mk(B, L, H, D), mk(B, L, H, D), mk(B, L, H, D), mk(H, 2 * A, D), mk(H, 2 * A, D)
    table = relative_offset_table(L, L, bucket_size=A, max_position=512, device=gpu)
    kk, pk = kernel_masks(_mask("mixed", B, L, H, g).to(gpu), B, L, L, gpu, segments_from_dense=False)
    assert kk is None and pk is not None
    scale = 1 / math.sqrt(3 * D)
    want, lse, _, _ = torch.ops.deberta_amd.dsa_fwd(q, k, v, kr, qr, table, kk, pk, A, scale, False)
    out, lse2 = torch.full_like(want, float("nan")), torch.full_like(lse, float("nan"))
    a = ops._fill_fwd_args(q, k, v, kr, qr, table, kk, pk, out, lse2, A, scale)
    _lib.check(lib.dsa_fwd(ctypes.byref(a), ctypes.c_void_p(torch.cuda.current_stream(gpu).cuda_stream)), "dsa_fwd")
    torch.cuda.synchronize(gpu)
    assert torch.equal(out, want)
    assert torch.equal(lse2, lse)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
def test_bytes_forward_bits_backward(dtype, gpu):
    """A forward on the mask's bytes (no workspace) of a call long enough for
    far blocks saves the bands everywhere; the backward takes the far blocks'
    terms from its own products and the saved bands elsewhere."""
    from deberta_amd import _lib, ops
    from deberta_amd.masks import kernel_masks
    from deberta_amd.relpos import relative_offset_table

    c = Case(B=1, H=2, L=600, D=64, buckets=32, max_pos=64, seed=12)
    x = make_inputs(c)
    x["mask"] = _mask("mixed", c.B, c.L, c.H, torch.Generator().manual_seed(c.seed))
    ref = oracle_run(c, x, dtype)
    q, k, v, kr, qr, dout = (x[n].to(gpu, dtype) for n in ("q", "k", "v", "kr", "qr", "dout"))
    table = relative_offset_table(c.L, c.L, bucket_size=c.buckets, max_position=c.max_pos, device=gpu)
    _, pk = kernel_masks(x["mask"].to(gpu), c.B, c.L, c.L, gpu, segments_from_dense=False)
    out = torch.empty_like(q)
    lse = torch.empty(c.B, c.H, c.L, device=gpu)
    bias = torch.empty(ops.bias_shape(q, k), dtype=ops.bias_dtype(dtype), device=gpu)
    scale = 1 / math.sqrt(3 * c.D)
    a = ops._fill_fwd_args(q, k, v, kr, qr, table, None, pk, out, lse, c.A, scale, bias)
    n = _lib.load().dsa_fwd_workspace_bytes(ctypes.byref(a))
    a.rel_saturated = 1 << 28
    assert n == _lib.load().dsa_fwd_workspace_bytes(ctypes.byref(a)) + 256  # far blocks are looked for
    a.rel_saturated = 0
    _lib.check(_lib.load().dsa_fwd(ctypes.byref(a), ctypes.c_void_p(torch.cuda.current_stream(gpu).cuda_stream)), "dsa_fwd")
    grads = torch.ops.deberta_amd.dsa_bwd(dout, q, k, v, kr, qr, table, None, pk, out, lse, bias, c.A, scale)
    got = dict(zip(("out", "dq", "dk", "dv", "dkr", "dqr"), [out, *grads]))
    for name, r in ref.items():
        g = got[name].float().cpu()
        err, tol = (max_rel(g, r), 1e-4) if dtype == torch.float32 else (min(max_rel(g, r), max_abs(g, r)), 2e-2)
        assert err <= tol, (name, err)
