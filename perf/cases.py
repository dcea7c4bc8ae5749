"""Timed cases of the fused disentangled attention and the blocks around it.

Each case is one call a user's program makes through the public entry points:
a serving pass of the attention layer, a training step (forward and backward)
of the attention on projected layers, of a whole encoder layer, or of the RTD
head with its loss.  ``listed()`` names the cases, ``draw`` gives more of the
same ranges, ``prepare`` builds what such a program holds before the call and
``run`` makes the call.  ``exact`` is the same call in float64 torch
operations, without this package.

Sizes follow the repository's own configurations (hidden 128 with 4 heads of
32; hidden 768 with 12 heads of 64; hidden 1024 with 16 heads; L = 512 padded
and unpadded, L = 4096 packed) and sizes between them, odd ones included.
"""

from __future__ import annotations

import math
import random
from types import SimpleNamespace

import torch
import torch.nn.functional as F

from deberta_amd import (
    DisentangledSelfAttention,
    FusedIntermediate,
    FusedOutput,
    FusedRTDHead,
    FusedSelfOutput,
    RelativeEmbeddings,
    SegmentMask,
    build_doc_block_mask,
    build_relative_position,
    disentangled_attention,
    get_attention_mask,
)

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
EPS = 1e-7  # the configurations' layer_norm_eps
# Standard deviation of q, k, v and the projected tables: N(0, 1) states (and
# a LayerNorm'd relative table) through N(0, 0.02) weights of hidden 768.
PROJECTED_STD = 0.02 * math.sqrt(768.0)


# ---------------------------------------------------------------------------
# the cases


def _attention(name, batch, heads, length, head_dim=64, dtype="bf16", mask="none", dropout=0.0, buckets=256, max_pos=512):
    """A training step of ``disentangled_attention`` on projected layers."""
    return {
        "name": name, "kind": "attention", "batch": batch, "heads": heads, "length": length, "head_dim": head_dim,
        "dtype": dtype, "mask": mask, "dropout": dropout, "buckets": buckets, "max_pos": max_pos,
    }


def _block(name, kind, batch, heads, length, head_dim, dtype, mask):
    """A pass of a module: ``serve`` (the attention layer's forward, without
    gradients), ``layer`` (one encoder layer's training step) or ``head``
    (the RTD head and its loss, training step)."""
    return {
        "name": name, "kind": kind, "batch": batch, "heads": heads, "length": length, "head_dim": head_dim,
        "dtype": dtype, "mask": mask, "dropout": 0.0, "buckets": 256, "max_pos": 512,
    }


def listed():
    return [
        # One attention layer of a small model, float32, two short sequences:
        # a call whose time is launches and host work.
        _block("serve_small_fp32", "serve", 2, 4, 128, 32, "fp32", "none"),
        # Serving a base-shaped model: an odd length, padded rows, bfloat16.
        _block("serve_base_ragged", "serve", 8, 12, 201, 64, "bf16", "key"),
        # The benchmark's step: base shape, full rows.
        _attention("train_base", 32, 12, 512),
        # The same shape with padded rows (lengths of a real batch).
        _attention("train_base_padded", 32, 12, 512, mask="key"),
        # Attention dropout on (the preset's 0.1), smaller batch.
        _attention("train_base_dropout", 12, 12, 512, dropout=0.1),
        # Packed long-context rows, documents given as ids.
        _attention("train_packed_ids", 4, 12, 4096, mask="docs"),
        # Packed rows with the reference's dense document mask.
        _attention("train_packed_dense", 6, 12, 1024, mask="docs_dense"),
        # A pairwise mask that is not made of documents: a local window with
        # one global token and padding.
        _attention("train_window", 4, 12, 1000, mask="window"),
        # Large shape, long unpadded rows.
        _attention("train_long", 4, 16, 2048),
        # Training without mixed precision.
        _attention("train_fp32", 4, 12, 384, dtype="fp32"),
        # One base encoder layer under bf16 autocast: attention, output and
        # FFN blocks, the shared relative table.
        _block("layer_base", "layer", 16, 12, 512, 64, "bf16", "key"),
        # The discriminator's head and loss under bf16 autocast.
        _block("head_base", "head", 16, 12, 512, 64, "bf16", "key"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    """One more case of the listed ones' ranges: the batch, length (odd ones
    among them), head count and head dim, type, mask and dropout of a
    training step or a module pass.  Costs no more than the largest listed
    case."""
    most = max(work(c)["flops"] for c in listed())
    while True:
        kind = rng.choice(["attention"] * 6 + ["serve"] * 2 + ["layer", "head"])
        heads, head_dim = rng.choice([(4, 32), (6, 64), (12, 64), (12, 64), (16, 64)])
        length = _log_int(rng, 48, 4096 if kind == "attention" else 768)
        if rng.random() < 0.5:
            length = max(64, length // 64 * 64)
        batch = min(64, max(1, _log_int(rng, 512, 40000) // length))
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp32"])
        mask, dropout = rng.choice(["none", "key"]), 0.0
        buckets, max_pos = 256, 512
        if kind == "attention":
            mask = rng.choice(["none", "key", "docs", "docs_dense", "window"])
            if rng.random() < 0.2:
                dropout = 0.1
            if rng.random() < 0.15:
                buckets, max_pos = rng.choice([(64, 512), (128, 512), (32, 256)])
        if kind in ("layer", "head"):
            dtype = "bf16"  # under autocast
        if dtype == "fp32":
            batch = max(1, batch // 4)  # float32 matrix rates are a fraction of bfloat16's
            length = min(length, 1024)
        case = {
            "kind": kind, "batch": batch, "heads": heads, "length": length, "head_dim": head_dim, "dtype": dtype,
            "mask": mask, "dropout": dropout, "buckets": buckets, "max_pos": max_pos,
        }
        dear = 16.0 if dtype == "fp32" else 1.0
        # a dense mask of no document form is visited whole
        pairs = 4.0 if mask in ("window", "docs", "docs_dense") else 1.0
        if work(case)["flops"] * dear * pairs <= most:
            return case


# ---------------------------------------------------------------------------
# inputs


def _span(case):
    return case["buckets"]


def _doc_mean(length):
    return min(600.0, length / 3.0)


def _window(length):
    return max(8, length // 16)


def _gen(seed, salt=0):
    return torch.Generator(device="cpu").manual_seed(int(seed) * 1000003 + salt)


def _key_keep(case, seed):
    """``(B, L)`` keep mask: a prefix of every row, the longest row full."""
    b, n = case["batch"], case["length"]
    lens = torch.randint(max(1, n // 8), n + 1, (b,), generator=_gen(seed, 1))
    lens[0] = n
    return torch.arange(n)[None, :] < lens[:, None]


def _doc_ids(case, seed):
    """``(B, L)`` document ids from 1, geometric lengths, the rows' tails
    padded (0)."""
    b, n = case["batch"], case["length"]
    g, mean = _gen(seed, 2), _doc_mean(case["length"])
    ids = torch.zeros(b, n, dtype=torch.int64)
    for r in range(b):
        end = n - int(torch.randint(0, max(2, n // 32), (1,), generator=g))
        pos, doc = 0, 1
        while pos < end:
            u = float(torch.rand((), generator=g, dtype=torch.float64))
            m = 1 + int(math.log1p(-u) / math.log1p(-1.0 / mean))
            ids[r, pos:min(pos + m, end)] = doc
            pos, doc = pos + m, doc + 1
    return ids


def _window_keep(case, seed):
    """``(B, L, L)`` keep mask: keys within the window, plus token 0 as key
    and as query, both tokens unpadded."""
    n, w = case["length"], _window(case["length"])
    i = torch.arange(n)
    near = (i[:, None] - i[None, :]).abs() <= w
    near[0, :] = True
    near[:, 0] = True
    k = _key_keep(case, seed)
    return near[None] & k[:, :, None] & k[:, None, :]


def _mask(case, seed):
    """The mask as a user's program passes it."""
    m = case["mask"]
    if m == "none":
        return None
    if m == "key":
        return get_attention_mask(_key_keep(case, seed).to(DEV))
    if m == "docs":
        return SegmentMask(_doc_ids(case, seed).to(device=DEV, dtype=torch.int32))
    if m == "docs_dense":
        return get_attention_mask(build_doc_block_mask(_doc_ids(case, seed).to(DEV)))
    return get_attention_mask(_window_keep(case, seed).to(DEV))


def _config(case):
    hidden = case["heads"] * case["head_dim"]
    return SimpleNamespace(
        hidden_size=hidden, num_attention_heads=case["heads"], intermediate_size=4 * hidden, share_att_key=True,
        pos_att_type="c2p|p2c", relative_attention=True, position_buckets=case["buckets"],
        max_relative_positions=case["max_pos"], max_position_embeddings=case["max_pos"], hidden_dropout_prob=0.0,
        attention_probs_dropout_prob=0.0, layer_norm_eps=EPS, norm_eps=EPS, hidden_act="gelu",
    )


def _fill(module, seed, dtype=torch.float32):
    """Weights N(0, 0.02), biases N(0, 0.02), LayerNorm weights near one."""
    g = _gen(seed, 3)
    with torch.no_grad():
        for name, p in module.named_parameters():
            x = torch.randn(p.shape, generator=g) * 0.02
            p.copy_(x + 1.0 if name.lower().endswith(("layernorm.weight", "norm.weight")) else x)
    return module.to(device=DEV, dtype=dtype)


class _Layer(torch.nn.Module):
    """One encoder layer and the encoder's shared relative table."""

    def __init__(self, cfg):
        super().__init__()
        self.rel = RelativeEmbeddings(cfg)
        self.attention = DisentangledSelfAttention(cfg)
        self.output = FusedSelfOutput(cfg)
        self.intermediate = FusedIntermediate(cfg)
        self.ffn_output = FusedOutput(cfg)

    def forward(self, x, mask, relative_pos):
        ctx, _ = self.attention(x, mask, relative_pos=relative_pos, rel_embeddings=self.rel())
        x = self.output(ctx, x)
        return self.ffn_output(self.intermediate(x), x)


def _states(case, seed):
    """What the exact computation and ``prepare`` share: float32 host tensors
    rounded to the case's type."""
    b, h, n, d = case["batch"], case["heads"], case["length"], case["head_dim"]
    dt, g = DTYPES[case["dtype"]], _gen(seed)
    rnd = lambda *s, std=1.0: (torch.randn(*s, generator=g) * std)
    if case["kind"] == "attention":
        r = 2 * _span(case)
        s = {"q": rnd(b, n, h * d, std=PROJECTED_STD), "k": rnd(b, n, h * d, std=PROJECTED_STD),
             "v": rnd(b, n, h * d, std=PROJECTED_STD), "kr": rnd(r, h * d, std=PROJECTED_STD),
             "qr": rnd(r, h * d, std=PROJECTED_STD), "dout": rnd(b, n, h * d)}
        return {k: t.to(dt) for k, t in s.items()}
    s = {"x": rnd(b, n, h * d)}
    if case["kind"] == "serve":
        s["x"] = s["x"].to(dt)
        s["rel"] = rnd(2 * _span(case), h * d).to(dt)
    elif case["kind"] == "layer":
        s["dout"] = rnd(b, n, h * d)
    else:
        s["labels"] = (torch.rand(b, n, generator=g) < 0.15).float()
    return s


def _module(case, seed):
    cfg = _config(case)
    if case["kind"] == "serve":
        return _fill(DisentangledSelfAttention(cfg), seed, DTYPES[case["dtype"]]).eval()
    return _fill(_Layer(cfg) if case["kind"] == "layer" else FusedRTDHead(cfg), seed).train()


def prepare(case, seed):
    s = {k: t.to(DEV) for k, t in _states(case, seed).items()}
    s["case"], s["mask"] = case, _mask(case, seed)
    if case["kind"] == "attention":
        for k in ("q", "k", "v", "kr", "qr"):
            s[k].requires_grad_(True)
        s["seed"] = int(seed)
        return s
    s["module"] = _module(case, seed)
    if case["kind"] == "serve":
        return s
    s["x"].requires_grad_(True)
    s["leaves"] = [s["x"], *s["module"].parameters()]
    if case["kind"] == "layer":  # the encoder hands its layers one matrix
        s["relative_pos"] = build_relative_position(
            case["length"], case["length"], bucket_size=case["buckets"], max_position=case["max_pos"], device=DEV
        )
    else:
        s["active"] = _key_keep(case, seed).to(DEV) if case["mask"] == "key" else None
    return s


# ---------------------------------------------------------------------------
# the call


def run(state):
    case = state["case"]
    if case["kind"] == "attention":
        return _run_attention(state, case)
    if case["kind"] == "serve":
        with torch.no_grad():
            out, _ = state["module"](state["x"], state["mask"], rel_embeddings=state["rel"])
        return out
    with torch.autocast("cuda", dtype=torch.bfloat16):
        if case["kind"] == "layer":
            out = state["module"](state["x"], state["mask"], state["relative_pos"])
            grad = state["dout"]
        else:
            loss, out = state["module"].forward_loss(state["x"], state["labels"], state["active"], state["mask"])
            grad = None
    grads = torch.autograd.grad(out if grad is not None else loss, state["leaves"], grad)
    return (out, *grads) if grad is not None else (loss.detach(), out, *grads)


def _run_attention(state, case):
    b, h, n, d = case["batch"], case["heads"], case["length"], case["head_dim"]
    if case["dropout"] > 0.0:  # the step's own random state: the same keep bits in every pass
        torch.random.default_generator.manual_seed(state["seed"])
    heads = lambda t: t.view(b, n, h, d)
    table = lambda t: t.view(-1, h, d).permute(1, 0, 2)
    out = disentangled_attention(
        heads(state["q"]), heads(state["k"]), heads(state["v"]), table(state["kr"]), table(state["qr"]),
        None, state["mask"], position_buckets=case["buckets"], max_relative_positions=case["max_pos"],
        att_type="c2p|p2c", layout="blhd", dropout_p=case["dropout"],
    )
    leaves = [state[k] for k in ("q", "k", "v", "kr", "qr")]
    grads = torch.autograd.grad(out, leaves, heads(state["dout"]))
    return (out.detach(), *grads)


# ---------------------------------------------------------------------------
# what a pass cannot do without


def _pairs(case):
    """(expected kept pairs of the batch, query rows that attend)."""
    b, n = case["batch"], case["length"]
    lo = max(1, n // 8)
    mean, mean2 = (lo + n) / 2.0, (lo * lo + lo * n + n * n) / 3.0
    if case["mask"] == "key":
        return b * mean2, b * mean
    if case["mask"] in ("docs", "docs_dense"):
        m = _doc_mean(n)  # geometric lengths cut at the row's end
        f = m / n
        per_token = 2.0 * m * (1.0 - f * (1.0 - math.exp(-1.0 / f)))
        return b * n * min(n, per_token), b * n
    if case["mask"] == "window":
        return b * mean * min(mean, 2 * _window(n) + 1), b * mean
    return float(b) * n * n, b * n


def _attention_flops(case):
    """Forward: scores and values over the kept pairs, and per relative term
    a dot product per query (key) and reachable table row."""
    pairs, rows = _pairs(case)
    rel = min(pairs, rows * min(2 * _span(case), 2 * case["length"] - 1))
    return 4.0 * case["heads"] * case["head_dim"] * (pairs + rel)


def work(case):
    b, h, n, d = case["batch"], case["heads"], case["length"], case["head_dim"]
    e = 2 if case["dtype"] == "bf16" else 4
    hid, r = h * d, 2 * _span(case)
    tok = b * n
    mask = {"none": 0, "key": tok, "docs": 4 * tok, "docs_dense": tok * n, "window": tok * n}[case["mask"]]
    attn = _attention_flops(case)
    if case["kind"] == "attention":
        return {"bytes": float(8 * tok * hid * e + 4 * r * hid * e + mask), "flops": 3.0 * attn}
    if case["kind"] == "serve":
        params = 3 * hid * hid + 3 * hid
        flops = 2.0 * tok * 3 * hid * hid + 2.0 * r * 2 * hid * hid + attn
        return {"bytes": float(2 * tok * hid * e + (params + r * hid) * e + mask), "flops": flops}
    if case["kind"] == "layer":  # float32 states and parameters, each read and its gradient written
        params = 3 * hid * hid + hid * hid + 8 * hid * hid + 13 * hid + r * hid
        gemms = 2.0 * tok * 12 * hid * hid + 2.0 * r * 2 * hid * hid
        return {"bytes": float(4 * (4 * tok * hid + 2 * params) + mask), "flops": 3.0 * (gemms + attn)}
    params = hid * hid + 4 * hid
    return {
        "bytes": float(4 * (2 * tok * hid + 2 * tok + 2 * params) + mask),
        "flops": 3.0 * (2.0 * tok * hid * hid + 2.0 * tok * hid),
    }


def tolerance(case):
    """About four times what the fused path shows against ``exact`` (2-norm
    per output): bfloat16 attention 0.0023 to 0.0028, float32 2.5e-7 to
    1.2e-6 by length, the autocast head 0.0039 and layer 0.0048."""
    if case["kind"] in ("attention", "serve"):
        return {"rel": 1.1e-2} if case["dtype"] == "bf16" else {"rel": 5e-6}
    return {"rel": 1.6e-2} if case["kind"] == "head" else {"rel": 2e-2}


# ---------------------------------------------------------------------------
# the same in float64


def _log_bucket(d, buckets, max_pos):
    """Log-bucketed relative position of integer offsets ``d``; float32 logs,
    as the models' configurations are trained with."""
    d = d.clamp(-max_pos + 1, max_pos - 1)
    mid = buckets // 2
    a = d.abs().clamp_min(1)
    base = math.log(max(max_pos - 1.0, mid + 1.0) / mid)
    far = torch.ceil(torch.log(a.float() / mid) / base * (mid - 1)) + mid
    return (torch.where(a < mid, a.float(), far) * torch.sign(d).float()).long()


def _philox(c0, c1, c2, c3, key):
    """Philox4x32-10 (Salmon et al., SC 2011) on int64 tensors holding
    32-bit words."""
    m = 0xFFFFFFFF
    k0, k1 = key & m, (key >> 32) & m
    for _ in range(10):
        p0, p1 = 0xD2511F53 * c0, 0xCD9E8D57 * c2  # modulo 2^64
        c0, c1, c2, c3 = ((p1 >> 32) & m) ^ c1 ^ k0, p1 & m, ((p0 >> 32) & m) ^ c3 ^ k1, p0 & m
        k0, k1 = (k0 + 0x9E3779B9) & m, (k1 + 0xBB67AE85) & m
    return c0, c1, c2, c3


def _drop_keep(case, row, seed):
    """Keep mask ``(H, L, L)`` of batch row ``row`` under the op's published
    dropout contract (dsa_dropout.h)."""
    h, n = case["heads"], case["length"]
    key = int(torch.randint(0, 1 << 62, (1,), dtype=torch.int64, generator=_plain_gen(seed)))
    t = int(round(case["dropout"] * 65536.0))
    tiles = (n + 63) // 64
    ar = lambda m: torch.arange(m, device=DEV, dtype=torch.int64)
    c0 = (ar(tiles)[:, None] * 8 + ar(8)[None, :]).view(1, 1, tiles, 8)
    shape = (h, n, tiles, 8)
    words = _philox(
        c0.expand(shape), ar(n).view(1, n, 1, 1).expand(shape), ar(h).view(h, 1, 1, 1).expand(shape),
        torch.full(shape, row, device=DEV, dtype=torch.int64), key,
    )
    u = torch.stack([x for wd in words for x in (wd & 0xFFFF, wd >> 16)], dim=-1)  # (.., 8, u = 4 kb + e)
    keep = (u >= t).view(h, n, tiles, 4, 2, 2, 4)  # g, half, kb, e
    keep = keep.permute(0, 1, 2, 4, 5, 3, 6).reshape(h, n, tiles * 64)  # key 16 (2 half + kb) + 4 g + e
    return keep[..., :n]


def _plain_gen(seed):
    return torch.Generator(device="cpu").manual_seed(int(seed))


def _keep_row(case, masks, row):
    """(``(L, L)`` keep mask or None, ``(L,)`` live rows or None) of one batch row."""
    m = case["mask"]
    if m == "none":
        return None, None
    if m == "key":
        # a key mask also marks the padded queries, whose rows are zero
        return masks[row][None, :].expand(case["length"], case["length"]), masks[row]
    if m == "window":
        return masks[row], masks[row].diagonal()
    ids = masks[row]
    return (ids[:, None] == ids[None, :]) & (ids != 0)[:, None], ids != 0


def _exact_masks(case, seed):
    m = case["mask"]
    if m == "none":
        return None
    make = {"key": _key_keep, "window": _window_keep}.get(m, _doc_ids)
    return make(case, seed).to(DEV)


def _attend_row(case, q, k, v, kr, qr, idx, keep, live, drop):
    """float64 attention of one batch row: q, k, v ``(H, L, D)``, tables
    ``(H, 2A, D)``."""
    d = case["head_dim"]
    top = 2 * _span(case) - 1
    h = case["heads"]
    c = (idx + _span(case)).clamp(0, top).expand(h, -1, -1)
    p = (-idx + _span(case)).clamp(0, top).expand(h, -1, -1)
    s = q @ k.transpose(1, 2)
    s = s + torch.gather(q @ kr.transpose(1, 2), 2, c)
    s = s + torch.gather(k @ qr.transpose(1, 2), 2, p.transpose(1, 2)).transpose(1, 2)
    s = s / math.sqrt(3.0 * d)
    if keep is not None:
        s = s.masked_fill(~keep, torch.finfo(torch.float32).min)
    prob = torch.softmax(s, dim=-1)
    if drop is not None:
        t = int(round(case["dropout"] * 65536.0))
        prob = prob * drop * (65536.0 / (65536.0 - t))
    o = prob @ v
    return o if live is None else o * live[None, :, None]


def _exact_attention(case, seed, q, k, v, kr, qr, dout=None):
    """(out, dq, dk, dv, dkr, dqr) or out alone; ``(B, L, H, D)`` layers and
    ``(2A, H, D)`` tables in float64, one batch row at a time."""
    n, span = case["length"], _span(case)
    masks = _exact_masks(case, seed)
    ar = torch.arange(n, device=DEV)
    idx = _log_bucket(ar[:, None] - ar[None, :], case["buckets"], case["max_pos"]).clamp(-span, span)
    hm = lambda t: t.permute(1, 0, 2).contiguous()
    outs, rows = [], []
    dkr = torch.zeros_like(hm(kr))
    dqr = torch.zeros_like(hm(qr))
    for b in range(case["batch"]):
        leaves = [hm(t).detach().requires_grad_(dout is not None) for t in (q[b], k[b], v[b], kr, qr)]
        keep, live = _keep_row(case, masks, b)
        drop = _drop_keep(case, b, seed) if case["dropout"] > 0.0 else None
        o = _attend_row(case, *leaves, idx, keep, live, drop)
        outs.append(o.detach().permute(1, 0, 2))
        if dout is not None:
            g = torch.autograd.grad(o, leaves, hm(dout[b]))
            rows.append([t.permute(1, 0, 2) for t in g[:3]])
            dkr += g[3]
            dqr += g[4]
    out = torch.stack(outs)
    if dout is None:
        return out
    return (out, *(torch.stack([r[i] for r in rows]) for i in range(3)), dkr.permute(1, 0, 2), dqr.permute(1, 0, 2))


class _ExactAttention(torch.autograd.Function):
    """The row-by-row float64 attention inside a float64 layer."""

    @staticmethod
    def forward(ctx, case, seed, q, k, v, kr, qr):
        ctx.save_for_backward(q, k, v, kr, qr)
        ctx.case, ctx.seed = case, seed
        return _exact_attention(case, seed, q, k, v, kr, qr)

    @staticmethod
    def backward(ctx, dout):
        with torch.enable_grad():
            g = _exact_attention(ctx.case, ctx.seed, *ctx.saved_tensors, dout)
        return (None, None, *g[1:])


def _exact_layer_attention(case, seed, w, x, rel):
    b, h, n, d = case["batch"], case["heads"], case["length"], case["head_dim"]
    lin = lambda name, t: F.linear(t, w[name + ".weight"], w[name + ".bias"])
    layers = [lin(nm, x).view(b, n, h, d) for nm in ("query_proj", "key_proj", "value_proj")]
    tables = [lin(nm, rel).view(-1, h, d) for nm in ("key_proj", "query_proj")]
    return _ExactAttention.apply(case, seed, *layers, *tables).reshape(b, n, h * d)


def _sub(w, prefix):
    return {k[len(prefix) + 1:]: t for k, t in w.items() if k.startswith(prefix + ".")}


def exact(case, seed):
    """``run``'s outputs for these inputs, in float64 torch operations.  The
    float32 cases' softmax, sums and products are all float64 here, so a
    result's distance from it is its rounding."""
    s = {k: t.to(DEV).double() for k, t in _states(case, seed).items()}
    b, h, n, d = case["batch"], case["heads"], case["length"], case["head_dim"]
    if case["kind"] == "attention":
        r = 2 * _span(case)
        res = _exact_attention(
            case, seed, *(s[k].view(b, n, h, d) for k in ("q", "k", "v")), *(s[k].view(r, h, d) for k in ("kr", "qr")),
            s["dout"].view(b, n, h, d),
        )
        return (res[0], *(t.reshape(b, n, h * d) for t in res[1:4]), *(t.reshape(r, h * d) for t in res[4:]))
    mod = _module(case, seed)
    w = {k: p.detach().double().requires_grad_(case["kind"] != "serve") for k, p in mod.named_parameters()}
    if case["kind"] == "serve":
        with torch.no_grad():
            return _exact_layer_attention(case, seed, w, s["x"], s["rel"])
    x = s["x"].requires_grad_(True)
    hid = h * d
    norm = lambda t, p: F.layer_norm(t, (hid,), w[p + ".weight"], w[p + ".bias"], EPS)
    lin = lambda t, p: F.linear(t, w[p + ".weight"], w[p + ".bias"])
    if case["kind"] == "layer":
        rel = F.layer_norm(w["rel.rel_embeddings.weight"], (hid,), w["rel.LayerNorm.weight"], w["rel.LayerNorm.bias"], EPS)
        a = _exact_layer_attention(case, seed, _sub(w, "attention"), x, rel)
        y = norm(lin(a, "output.dense") + x, "output.LayerNorm")
        out = norm(lin(F.gelu(lin(y, "intermediate.dense")), "ffn_output.dense") + y, "ffn_output.LayerNorm")
        return (out.detach(), *torch.autograd.grad(out, [x, *w.values()], s["dout"]))
    z = F.gelu(lin(norm(x + x[:, :1], "norm"), "dense"))
    logits = lin(z, "classifier").squeeze(-1)
    act = _key_keep(case, seed).to(DEV).double() if case["mask"] == "key" else torch.ones(b, n, device=DEV, dtype=torch.float64)
    per = F.binary_cross_entropy_with_logits(logits, s["labels"], reduction="none")
    loss = (per * act).sum() / act.sum().clamp(min=1.0)
    return (loss.detach(), logits.detach(), *torch.autograd.grad(loss, [x, *w.values()]))
