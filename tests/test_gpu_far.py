"""Far blocks: 128 x 128 blocks of (query, key) pairs whose relative position
has saturated, run without bands (FarSpan, dsa_tiles.h) where a call has
enough of them (far_call, dsa_launch.h).  The op against the
CPU oracle where the rule or the span can go wrong: extents on both sides of
the rule, a span on one side only, past the last query or key block or
nowhere, every mask form that takes it, dropout and the p2p query rows; and
the backward in separate stage calls against the one call.  The bounds are the
parity suite's (fp32 1e-4 of scale, bf16 2e-2)."""

from __future__ import annotations

import ctypes
import math

import pytest
import torch

from tests._cases import Case, make_inputs
from tests.test_gpu_parity import _check

pytestmark = pytest.mark.gpu

_CASES = [
    Case(B=1, H=2, L=256, D=64, buckets=-1, max_pos=1, seed=1),  # saturated beside the diagonal, 2 blocks
    Case(B=2, H=2, L=384, D=64, buckets=32, max_pos=64, seed=2),  # first length past the rule (129 >= 64)
    Case(B=1, H=2, L=385, D=32, buckets=32, max_pos=64, seed=3),  # one row in the last block
    Case(B=1, H=1, L=700, D=64, buckets=64, max_pos=512, seed=4),  # looked for, hardly any found
    Case(B=1, H=1, L=450, D=64, buckets=64, max_pos=4096, seed=5),  # looked for, none found
    Case(B=2, H=1, L=90, Lk=700, D=64, buckets=32, max_pos=64, seed=6),  # key side only, one query block
    Case(B=2, H=1, L=700, Lk=90, D=32, buckets=32, max_pos=64, seed=7),  # query side only
    Case(B=1, H=2, L=641, D=64, buckets=32, max_pos=64, types="c2p", seed=8),
    Case(B=1, H=2, L=641, D=64, buckets=32, max_pos=64, types="p2c", seed=9),
    Case(B=1, H=2, L=640, D=64, buckets=-1, max_pos=64, types="c2p|p2c|p2p", seed=10),
    Case(B=3, H=2, L=600, D=64, buckets=32, max_pos=64, mask="key", seed=11),
    Case(B=2, H=2, L=900, D=64, buckets=32, max_pos=64, mask="seg", seed=12),
    Case(B=2, H=2, L=520, D=32, buckets=32, max_pos=64, mask="seg_mixed", seed=13),
    Case(B=2, H=2, L=500, D=64, buckets=32, max_pos=64, mask="dead", seed=14),
    Case(B=1, H=2, L=600, D=64, buckets=32, max_pos=64, dropout=0.1, seed=15),
    Case(B=2, H=1, L=700, D=64, buckets=32, max_pos=64, mask="seg", dropout=0.1, seed=16),
    Case(B=1, H=2, L=512, D=64, buckets=-1, max_pos=1, seed=17),  # saturated beside the diagonal, 4 blocks
    Case(B=2, H=2, L=700, D=32, buckets=32, max_pos=64, mask="seg_mixed", seed=18),
]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("c", _CASES, ids=[str(c.seed) for c in _CASES])
def test_far_blocks(c, dtype, gpu):
    # a saturated table row sums nearly all pairs of a head: its bf16
    # gradient is held to its scale
    _check(c, dtype, gpu, grads_to_scale=True)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("p2p", [False, True])
@pytest.mark.parametrize("Lq,Lk", [(640, 640), (130, 900)])
def test_far_stage_split(Lq, Lk, p2p, dtype, gpu):
    """PREP, DKDV, DQ, TABLE and SUM in calls of their own (the table kernel
    then sums the far blocks' dKr itself) and DQ|TABLE in one, against one
    call for all."""
    from deberta_amd import _lib, ops
    from deberta_amd.attention import relative_operands
    from deberta_amd.relpos import relative_offset_table

    lib = _lib.load()
    B, H, D, A = 2, 2, 64, 32
    g = torch.Generator().manual_seed(5)
    mk = lambda *s: torch.randn(*s, generator=g).to(gpu, dtype)
    q, k, v, dout = mk(B, Lq, H, D), mk(B, Lk, H, D), mk(B, Lk, H, D), mk(B, Lq, H, D)
    kr, qr = mk(H, 2 * A, D), mk(H, 2 * A, D)
    table = relative_offset_table(Lq, Lk, bucket_size=A, max_position=64, device=gpu)
    qc = relative_operands(["c2p", "p2c", "p2p"], q, kr, qr, A)[2].contiguous() if p2p else None
    scale = 1 / math.sqrt(D * 3)
    out, lse, bias, aux = torch.ops.deberta_amd.dsa_fwd(q, k, v, kr, qr, table, None, None, A, scale, True, qc)
    stream = ctypes.c_void_p(torch.cuda.current_stream(gpu).cuda_stream)
    bits = {n: getattr(_lib, f"DSA_STAGE_{n}") for n in ("PREP", "DQ", "DKDV", "TABLE", "SUM")}

    def run(calls):
        grads = [torch.full_like(t, float("nan")) for t in (q, k, v)]
        dqc = torch.full_like(q, float("nan")) if p2p else None
        tabs = [torch.zeros((H, 2 * A, D), dtype=torch.float32, device=gpu) for _ in range(2)]
        a = ops.fill_bwd_args(dout, q, k, v, kr, qr, table, None, None, out, lse, bias, A, scale, *grads, *tabs,
                              qc=qc, dqc=dqc, dropout_bits=aux)
        ws = torch.empty((ops.bwd_workspace_bytes(a),), dtype=torch.uint8, device=gpu)
        a.workspace, a.workspace_bytes = ws.data_ptr(), ws.numel()
        for c in calls:
            a.stages = sum(bits[s] for s in c.split("|") if s)
            _lib.check(lib.dsa_bwd(ctypes.byref(a), stream), "dsa_bwd")
        torch.cuda.synchronize(gpu)
        return dict(zip(["dq", "dk", "dv", "dkr", "dqr", "dqc"], grads + tabs + [dqc]))

    ref = run([""])
    # the far rows are summed from float32 row sums of dS in one call and from
    # its products in the other: fp32 sums in another order, and for bf16 the
    # same products of bf16 dS
    for calls in (["PREP", "DKDV", "DQ", "TABLE", "SUM"], ["PREP", "DKDV", "DQ|TABLE", "SUM"]):
        got = run(calls)
        for name, b in ref.items():
            if b is None:
                continue
            assert torch.isfinite(got[name]).all(), name
            if name in ("dkr", "dqr"):
                err = float((got[name] - b).abs().max() / b.abs().max())
                assert err <= 1e-5, (calls, name, err)
            else:
                assert torch.equal(got[name], b), (calls, name)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("types", ["c2p|p2c", "c2p", "p2c"])
@pytest.mark.parametrize("mask", ["none", "key"])
def test_far_table_not_monotone(mask, types, dtype, gpu):
    """A table that comes back to its end's rows on every block diagonal but
    not on the offsets between them has no far block: out, dq, dk and dv are
    those of any Toeplitz table (dkr and dqr need a monotone one).  The forward
    without a workspace searches in its workgroups: equal to the last bit."""
    from deberta_amd import _lib, ops
    from deberta_amd.masks import kernel_masks
    from oracle import eager

    c = Case(B=2, H=2, L=514, D=64, buckets=32, max_pos=64, mask=mask, types=types, seed=21)
    x = make_inputs(c)
    d = torch.arange(-(c.L - 1), c.L)
    table = (d + 32) % 64 - 32
    i = torch.arange(c.L)
    leaf = lambda t: t.to(dtype).float().requires_grad_()
    hm = lambda t: t.permute(0, 2, 1, 3)
    rq, rk, rv = (leaf(x[n]) for n in ("q", "k", "v"))
    rkr, rqr = (leaf(x[n]) if t in c.type_list else None for n, t in (("kr", "c2p"), ("qr", "p2c")))
    ctx, _ = eager.attend(
        hm(rq), hm(rk), hm(rv), rkr, rqr, table[i[:, None] - i[None] + c.L - 1], x["mask"], types=c.type_list,
        att_span=c.A, use_relative=True,
    )
    ref = [ctx, *torch.autograd.grad(ctx, [rq, rk, rv], hm(x["dout"].to(dtype).float()))]

    q, k, v = (x[n].to(gpu, dtype).requires_grad_() for n in ("q", "k", "v"))
    kr, qr = (x[n].to(gpu, dtype).requires_grad_() if t in c.type_list else None for n, t in (("kr", "c2p"), ("qr", "p2c")))
    rel = table.to(gpu, torch.int32)
    kk, _ = kernel_masks(None if x["mask"] is None else x["mask"].to(gpu), c.B, c.L, c.L, gpu)
    scale = 1 / math.sqrt((1 + len(c.type_list)) * c.D)
    out, lse, _, _ = torch.ops.deberta_amd.dsa_fwd(q, k, v, kr, qr, rel, kk, None, c.A, scale, True)
    got = [hm(out), *torch.autograd.grad(out, [q, k, v], x["dout"].to(gpu, dtype))]
    for name, a, b in zip(("out", "dq", "dk", "dv"), got, ref):
        err = float((a.detach().float().cpu() - b).abs().max())
        tol = 2e-2 if dtype == torch.bfloat16 else 1e-4 * float(b.abs().max())
        assert err <= tol, (name, err)

    out2, lse2 = torch.full_like(out, float("nan")), torch.full_like(lse, float("nan"))
    a = ops._fill_fwd_args(q, k, v, kr, qr, rel, kk, None, out2, lse2, c.A, scale)
    _lib.check(_lib.load().dsa_fwd(ctypes.byref(a), ctypes.c_void_p(torch.cuda.current_stream(gpu).cuda_stream)), "dsa_fwd")
    torch.cuda.synchronize(gpu)
    assert torch.equal(out2, out) and torch.equal(lse2, lse)


def _grads(c: Case, x: dict, dtype, gpu):
    """(out, dq, dk, dv, dkr, dqr) of the op on the case's inputs."""
    from deberta_amd import ops  # noqa: F401
    from deberta_amd.masks import SegmentMask, kernel_masks
    from deberta_amd.relpos import relative_offset_table

    q, k, v, kr, qr = (x[n].to(gpu, dtype).requires_grad_() for n in ("q", "k", "v", "kr", "qr"))
    table = relative_offset_table(c.L, c.L, bucket_size=c.buckets, max_position=c.max_pos, device=gpu)
    mask = SegmentMask(x["seg"]) if x["seg"] is not None else x["mask"].to(gpu)
    kk, pk = kernel_masks(mask, c.B, c.L, c.L, gpu, segments_from_dense=False)
    out = torch.ops.deberta_amd.dsa_fwd(q, k, v, kr, qr, table, kk, pk, c.A, 1 / math.sqrt(3 * c.D), True)[0]
    return [out.detach(), *torch.autograd.grad(out, [q, k, v, kr, qr], x["dout"].to(gpu, dtype))]


def _padded(c: Case, live: int, kind: str) -> dict:
    """The case's inputs with queries and keys past ``live`` padded, as a key
    mask, segment ids or a pair mask."""
    x = make_inputs(c)
    keep = (torch.arange(c.L) < live)[None].repeat(c.B, 1)
    if kind == "key":
        x["mask"] = keep[:, None, None, :]
    elif kind == "seg":
        x["seg"] = keep.long()
    else:
        x["mask"] = (keep[:, :, None] & keep[:, None, :])[:, None]
    return x


def _same(got, want):
    for name, a, b in zip(("out", "dq", "dk", "dv", "dkr", "dqr"), got, want):
        assert torch.isfinite(a).all(), name
        if name in ("dkr", "dqr"):  # sums of atomic additions: one step of the dtype, 2^-20 of scale in fp32
            tol = (2.0**-20 if a.dtype == torch.float32 else 2.0**-7) * float(b.float().abs().max())
            assert float((a.float() - b.float()).abs().max()) <= tol, name
        else:
            assert torch.equal(a, b), name


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("kind", ["key", "seg", "pair"])
def test_far_dead_rows_overflow(kind, dtype, gpu):
    """Padded query rows whose products with the tables overflow, beside live
    ones of the same 32 rows, change nothing: as with zeros there."""
    c = Case(B=2, H=2, L=768, D=64, buckets=32, max_pos=64, seed=22)
    x = _padded(c, 530, kind)
    x["q"][:, 530:] = 0
    want = _grads(c, x, dtype, gpu)
    x["q"][:, 530:] = 3e38
    _same(_grads(c, x, dtype, gpu), want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("kind", ["key", "seg", "pair"])
def test_far_dead_chunks(kind, dtype, gpu):
    """What the padded queries of 32-row chunks without a live one hold (NaN)
    reaches nothing, the far rows of dKr included."""
    c = Case(B=2, H=2, L=768, D=64, buckets=32, max_pos=64, seed=23)
    x = _padded(c, 544, kind)
    for n in ("q", "dout"):
        x[n][:, 544:] = 0
    want = _grads(c, x, dtype, gpu)
    for n in ("q", "dout"):
        x[n][:, 544:] = float("nan")
    _same(_grads(c, x, dtype, gpu), want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
def test_far_side_without_pairs(dtype, gpu):
    """Far keys on one side only: the other side's table rows reach nothing."""
    c = Case(B=1, H=2, L=800, D=64, buckets=64, max_pos=256, seed=24)
    x = make_inputs(c)
    x["mask"] = torch.ones(c.L, c.L, dtype=torch.bool).triu()[None, None]
    x["kr"][:, 2 * c.A - 1] = 0
    x["qr"][:, 1] = 0  # (bucket A - 1)
    want = _grads(c, x, dtype, gpu)
    x["kr"][:, 2 * c.A - 1] = float("nan")
    x["qr"][:, 1] = float("nan")
    _same(_grads(c, x, dtype, gpu), want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), float("-inf")])
def test_far_term_not_finite(value, dtype, gpu):
    """A far c2p term that is not finite stays with the pairs it belongs to:
    the rows of the same tiles whose far pairs are all masked are as without
    it."""
    from deberta_amd import ops  # noqa: F401
    from deberta_amd.masks import kernel_masks
    from deberta_amd.relpos import relative_offset_table

    c = Case(B=1, H=2, L=700, D=64, buckets=32, max_pos=64, types="c2p", seed=25)
    x = make_inputs(c)
    i = torch.arange(c.L)
    keep = (i[:, None] - i[None]).abs() <= 20  # none of these reads a saturated row
    keep[::128] = True  # one row of every tile keeps all keys
    kk, pk = kernel_masks(keep[None, None].to(gpu), c.B, c.L, c.L, gpu, segments_from_dense=False)
    table = relative_offset_table(c.L, c.L, bucket_size=c.buckets, max_position=c.max_pos, device=gpu)
    q, k, v = (x[n].to(gpu, dtype) for n in ("q", "k", "v"))
    local = torch.arange(c.L) % 128 != 0
    got = []
    for far in (0.0, value):
        kr = x["kr"].clone()
        kr[:, 1] = 0.0  # the row of the keys far after the queries (bucket 1 - A)
        kr[:, 1, 0] = far
        out, lse, _, _ = torch.ops.deberta_amd.dsa_fwd(
            q, k, v, kr.to(gpu, dtype), None, table, kk, pk, c.A, 1 / math.sqrt(2 * c.D), False
        )
        got.append((out[:, local], lse[:, :, local]))
    assert torch.isfinite(got[0][0]).all()
    for a, b in zip(*got):
        assert torch.equal(a, b)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("dropout", [0.0, 0.1])
@pytest.mark.parametrize("types", ["c2p|p2c", "c2p|p2c|p2p"])
@pytest.mark.parametrize("mask", ["none", "key", "seg", "pair"])
def test_far_kernels(mask, types, dropout, D, dtype, gpu):
    """Every form of the kernels with far blocks (66% of the blocks here)."""
    c = Case(B=1, H=2, L=900, D=D, buckets=32, max_pos=64, types=types, mask=mask, dropout=dropout, seed=26)
    _check(c, dtype, gpu, grads_to_scale=True)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("hint", [1, 100, 1 << 20])
def test_far_hint(hint, dtype, gpu):
    """What a caller says of the saturation (here at 255) decides the kernels
    that run, not what they compute: too near, too far, none."""
    from deberta_amd import ops  # noqa: F401
    from deberta_amd.relpos import relative_offset_table

    c = Case(B=1, H=2, L=700, D=64, buckets=64, max_pos=256, seed=27)
    x = make_inputs(c)
    table = relative_offset_table(c.L, c.L, bucket_size=c.buckets, max_position=c.max_pos, device=gpu)
    runs = []
    for h in (0, hint):
        q, k, v, kr, qr = (x[n].to(gpu, dtype).requires_grad_() for n in ("q", "k", "v", "kr", "qr"))
        out = torch.ops.deberta_amd.dsa_fwd(
            q, k, v, kr, qr, table, None, None, c.A, 1 / math.sqrt(3 * c.D), True, None, 0, None, h
        )[0]
        runs.append([out.detach(), *torch.autograd.grad(out, [q, k, v, kr, qr], x["dout"].to(gpu, dtype))])
    # far terms are fp32 sums where the bands are rounded (fp16 for bf16)
    tol = 1e-5 if dtype == torch.float32 else 1e-2
    for name, a, b in zip(("out", "dq", "dk", "dv", "dkr", "dqr"), *runs):
        assert float((a.float() - b.float()).norm()) <= tol * float(a.float().norm()), name


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("kind", ["key", "seg", "pair"])
def test_far_stage_split_masked(kind, dtype, gpu):
    """The dq kernel alone, whose key tiles a mask lists, with far blocks:
    DKDV, DQ, TABLE and SUM in calls of their own against one call."""
    from deberta_amd import _lib, ops
    from deberta_amd.masks import SegmentMask, kernel_masks
    from deberta_amd.relpos import relative_offset_table

    c = Case(B=2, H=2, L=768, D=64, buckets=32, max_pos=64, seed=28)
    x = _padded(c, 700, kind)
    q, k, v, kr, qr, dout = (x[n].to(gpu, dtype) for n in ("q", "k", "v", "kr", "qr", "dout"))
    table = relative_offset_table(c.L, c.L, bucket_size=c.buckets, max_position=c.max_pos, device=gpu)
    mask = SegmentMask(x["seg"]) if x["seg"] is not None else x["mask"].to(gpu)
    kk, pk = kernel_masks(mask, c.B, c.L, c.L, gpu, segments_from_dense=False)
    scale = 1 / math.sqrt(3 * c.D)
    out, lse, bias, aux = torch.ops.deberta_amd.dsa_fwd(q, k, v, kr, qr, table, kk, pk, c.A, scale, True)
    stream = ctypes.c_void_p(torch.cuda.current_stream(gpu).cuda_stream)
    runs = []
    for calls in ([""], ["PREP", "DKDV", "DQ", "TABLE", "SUM"]):
        grads = [torch.full_like(t, float("nan")) for t in (q, k, v)]
        tabs = [torch.zeros((c.H, 2 * c.A, c.D), dtype=torch.float32, device=gpu) for _ in range(2)]
        a = ops.fill_bwd_args(dout, q, k, v, kr, qr, table, kk, pk, out, lse, bias, c.A, scale, *grads, *tabs,
                              dropout_bits=aux)
        ws = torch.empty((ops.bwd_workspace_bytes(a),), dtype=torch.uint8, device=gpu)
        a.workspace, a.workspace_bytes = ws.data_ptr(), ws.numel()
        for n in calls:
            a.stages = getattr(_lib, f"DSA_STAGE_{n}") if n else 0
            _lib.check(_lib.load().dsa_bwd(ctypes.byref(a), stream), "dsa_bwd")
        torch.cuda.synchronize(gpu)
        runs.append(grads + tabs)
    for name, a, b in zip(("dq", "dk", "dv", "dkr", "dqr"), *runs):
        if name in ("dkr", "dqr"):  # fp32 sums in another order
            assert float((a - b).abs().max()) <= 1e-5 * float(a.abs().max()), name
        else:
            assert torch.isfinite(a).all() and torch.equal(a, b), name
