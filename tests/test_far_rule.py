"""The rule that sends a call to the kernels with far blocks (far_call,
dsa_launch.h), read from the forward's workspace, whose last 256 bytes then
hold their span: against the share of far blocks counted block by block."""

from __future__ import annotations

import ctypes

import pytest

from deberta_amd import _lib
from deberta_amd.relpos import relative_offset_table, saturation_distance


def _looks(Lq, Lk, A, sat=0, dtype=None, seg=False, qc=False, drop=0):
    lib = _lib.load()
    a = _lib.DsaFwdArgs()
    a.B, a.H, a.Lq, a.Lk, a.D, a.att_span = 1, 1, Lq, Lk, 64, A
    a.dtype = _lib.DSA_BF16 if dtype is None else dtype
    a.flags, a.rel_saturated, a.dropout_threshold = _lib.DSA_C2P | _lib.DSA_P2C, sat, drop
    buf = ctypes.create_string_buffer(16)
    p = ctypes.cast(buf, ctypes.c_void_p).value
    a.dropout_bits = p  # (the caller's: none in the workspace)
    if seg:
        a.seg = p
    if qc:
        a.qc = p
    n = lib.dsa_fwd_workspace_bytes(ctypes.byref(a))
    a.rel_saturated = 1 << 28  # never
    return n - lib.dsa_fwd_workspace_bytes(ctypes.byref(a)) == 256


def _share(Lq, Lk, sat):
    nq, nk = (Lq + 127) // 128, (Lk + 127) // 128
    far = sum(
        1 for i in range(nq) for j in range(nk) for d in (i - j, j - i) if d >= 1 and 128 * d - 127 >= sat
    )
    return far, far / (nq * nk)


@pytest.mark.parametrize(
    "form,need",
    [
        (dict(), 0.25), (dict(drop=6554), 0.25), (dict(qc=True), 0.34), (dict(seg=True), 0.5),
        (dict(seg=True, drop=6554), 0.6), (dict(dtype=_lib.DSA_F32), 0.1), (dict(dtype=_lib.DSA_F32, seg=True), 0.3),
        (dict(dtype=_lib.DSA_F32, qc=True), 0.1),
    ],
)
def test_rule(form, need):
    for Lq, Lk in [(n, n) for n in range(1, 4200, 129)] + [(70, 900), (900, 70), (1, 4096), (2500, 700)]:
        for sat in (1, 2, 63, 64, 127, 128, 129, 255, 256, 511, 2000):
            far, share = _share(Lq, Lk, sat)
            assert _looks(Lq, Lk, 32, sat, **form) == (far > 0 and share >= need - 1e-9), (Lq, Lk, sat, share)
            if sat % 2 == 0:  # unknown: twice att_span
                assert _looks(Lq, Lk, sat // 2, **form) == (far > 0 and share >= need - 1e-9), (Lq, Lk, sat, share)


def test_largest_hint():
    assert not _looks(4096, 4096, 32, 2**31 - 1)


@pytest.mark.parametrize("buckets,max_pos", [(256, 512), (64, 512), (32, 64), (-1, 64), (2, 64), (8, 4), (24, 2)])
def test_saturation_distance(buckets, max_pos):
    """No offset past the distance reads another row than the last one."""
    A = buckets if buckets > 0 else max_pos
    L = 2 * max_pos + 3
    rows = relative_offset_table(L, L, bucket_size=buckets, max_position=max_pos).clamp(-A, A)
    c2p = (rows + A).clamp(0, 2 * A - 1)
    p2c = (A - rows).clamp(0, 2 * A - 1)
    sat = saturation_distance(buckets, max_pos, A)
    for t in (c2p, p2c):
        assert (t[L - 1 + sat:] == t[-1]).all() and (t[: L - sat] == t[0]).all()
