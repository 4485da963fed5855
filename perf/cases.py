"""Performance cases of neighbourhood attention: what programs built on this
package have it do, through its public entry points.

A case is a dict of plain values; a size, kernel or dilation is a text with
one number per axis ("56x56"), causal axes a text of 0/1 per axis.  ``op``
names the entry points:

* ``na``: ``na{1,2,3}d`` (forward, or forward and gradients), with GQA
  (``kv_heads`` < ``heads``), strided queries, and q/k/v either separate
  tensors or views of one packed projection (``packed``);
* ``split``: ``na{r}d_qk`` -> softmax -> ``na{r}d_av``, with gradients;
* ``rpb``: ``extras.allin1`` logits with a relative position bias -> softmax
  -> AV, with gradients (the bias's among them);
* ``varlen``: ``na{r}d_varlen`` on a padded batch, with gradients;
* ``extra``: ``na{r}d`` with ``additional_keys`` / ``additional_values``,
  with gradients;
* ``module``: a ``NeighborhoodAttention{r}D`` layer, with the gradients of
  its input and parameters.

``exact`` restates every op in float64 torch: window indices per axis, then a
loop over the window's entries.
"""
from __future__ import annotations

import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "natten-mps_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import natten_mps_amd as na  # noqa: E402
from natten_mps_amd.extras import allin1  # noqa: E402

_DEFAULTS = dict(op="na", dtype="bfloat16", batch=1, size="56x56", heads=4, kv_heads=0, dim=32, kernel="7x7",
                 dilation="1x1", stride=1, causal="00", grad=True, packed=False, tokens=0)


def _case(**over):
    c = dict(_DEFAULTS, **over)
    rank = len(_ints(c["size"]))
    for key, one in (("dilation", "x".join("1" * rank)), ("causal", "0" * rank)):
        if key not in over:
            c[key] = one
    c["kv_heads"] = c["kv_heads"] or c["heads"]
    return c


def _ints(text):
    return tuple(int(x) for x in text.split("x"))


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------


def listed():
    return [
        # the smallest call: one short sequence layer in single precision, no
        # gradients; its time is latency and launches
        _case(name="line_fp32_forward", dtype="float32", batch=2, size="128", heads=4, dim=32, kernel="7",
              grad=False),
        # a small single-precision training step, causal on one axis
        _case(name="plane_fp32_step", dtype="float32", batch=2, size="32x32", heads=4, dim=32, kernel="7x7",
              causal="10"),
        # the first level of an image backbone at a training batch
        _case(name="plane_bf16_step", batch=64, size="56x56", heads=4, dim=32, kernel="7x7"),
        # inference on a few large images of an odd size, the largest call:
        # wide windows, half precision, q/k/v as views of the packed projection
        _case(name="plane_fp16_forward", dtype="float16", batch=4, size="135x241", heads=8, dim=64,
              kernel="13x13", grad=False, packed=True),
        # long sequences with grouped kv heads, causal: a language-model layer
        _case(name="line_gqa_causal_step", batch=4, size="16384", heads=8, kv_heads=2, dim=64, kernel="33",
              causal="1"),
        # video: a 3-D layer with a kernel and dilation of its own per axis
        _case(name="volume_bf16_step", batch=2, size="16x32x32", heads=8, dim=64, kernel="3x7x7",
              dilation="1x2x2"),
        # the split ops, for programs that work on the attention weights
        # between QK and AV
        _case(name="split_bf16_step", op="split", batch=16, size="56x56", heads=4, dim=32, kernel="7x7"),
        # the same in single precision on a ragged size, dilated
        _case(name="split_fp32_step", op="split", dtype="float32", batch=4, size="45x61", heads=4, dim=32,
              kernel="7x7", dilation="2x2"),
        # relative position bias at an image backbone's first level
        _case(name="rpb_bf16_step", op="rpb", batch=16, size="56x56", heads=4, dim=32, kernel="7x7"),
        # images of mixed sizes in one padded batch
        _case(name="varlen_bf16_step", op="varlen", batch=16, size="56x56", heads=4, dim=32, kernel="7x7"),
        # an image layer whose queries attend to extra (register) tokens too
        _case(name="extra_bf16_step", op="extra", batch=8, size="48x48", heads=8, dim=64, kernel="7x7", tokens=16),
        # a whole layer of a backbone's second level: projections and
        # attention on their packed output
        _case(name="module_bf16_step", op="module", batch=32, size="28x28", heads=8, dim=32, kernel="7x7",
              dilation="2x2"),
    ]


# Sizes that a draw keeps under: q elements, and window entries times the
# head dim over all queries (less of both in single precision).
_MOST_ELEMENTS = 16 << 20
_MOST_PAIR_DIMS = 1_200_000_000


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        c = _draw_one(rng)
        if c is not None:
            return c


def _draw_one(rng):
    op = rng.choice(("na", "na", "na", "na", "split", "split", "rpb", "varlen", "extra", "module"))
    rank = {"rpb": rng.choice((1, 2, 2))}.get(op) or rng.choice((1, 2, 2, 2, 3))
    dtype = rng.choice(("bfloat16", "bfloat16", "float16", "float32"))
    dim = rng.choice((32, 32, 64, 64, 128))
    heads = rng.choice((1, 2, 3, 4, 6, 8, 12))
    if rank == 1:
        size = (_log_int(rng, 64, 16384),)
        kernel = (rng.choice((3, 7, 9, 15, 33, 63)),)
        dilation = (rng.choice((1, 1, 1, 2, 4, 8)),)
    elif rank == 2:
        size = tuple(_log_int(rng, 14, 256) for _ in range(2))
        k = rng.choice((3, 5, 7, 7, 7, 9, 11, 13))
        kernel = (k, k)
        d = rng.choice((1, 1, 1, 2, 3, 4))
        dilation = (d, d)
    else:
        size = (_log_int(rng, 4, 24),) + tuple(_log_int(rng, 12, 64) for _ in range(2))
        k = rng.choice((3, 5, 7))
        kernel = (rng.choice((3, 3, 5)), k, k)
        d = rng.choice((1, 1, 2))
        dilation = (1, d, d)
    grad = op != "na" or rng.random() < 0.7
    kv_heads, stride, causal, packed, tokens = heads, 1, (0,) * rank, False, 0
    if op == "na":
        turn = rng.random()
        if turn < 0.2 and heads % 2 == 0:
            kv_heads = heads // 2
        elif turn < 0.4:
            packed = True
        elif turn < 0.5 and max(dilation) == 1 and dtype != "float32":
            stride = 2
        if rng.random() < 0.25:
            causal = (1,) + (0,) * (rank - 1)
    if op == "extra":
        tokens = rng.choice((1, 4, 16, 77))
    if op in ("split", "rpb", "varlen", "extra", "module") and dtype == "float32" and dim == 128:
        dim = 64
    # a window has to fit its axis with room to move in
    if any(n < k * d + 1 for n, k, d in zip(size, kernel, dilation)):
        return None
    share = 1.0 if dtype != "float32" else 0.06 if op in ("split", "rpb") else 0.25
    per = heads * dim * math.prod(size)
    most = min(_MOST_ELEMENTS, _MOST_PAIR_DIMS / math.prod(kernel)) * share
    if per > most:
        return None
    batch = _log_int(rng, 1, min(64, int(most / per)))
    return _case(op=op, dtype=dtype, batch=batch, size="x".join(map(str, size)), heads=heads, kv_heads=kv_heads,
                 dim=dim, kernel="x".join(map(str, kernel)), dilation="x".join(map(str, dilation)), stride=stride,
                 causal="".join(map(str, causal)), grad=grad, packed=packed, tokens=tokens)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------


def _params(case):
    size, kernel, dilation = _ints(case["size"]), _ints(case["kernel"]), _ints(case["dilation"])
    causal = tuple(x == "1" for x in case["causal"])
    return size, kernel, dilation, causal


def _extents(case, seed):
    """Per-sample extents of a padded batch: half of each axis to all of it,
    the first sample at full size."""
    size, kernel, dilation, _ = _params(case)
    g = torch.Generator().manual_seed(seed + 17)
    rows = [size]
    for _ in range(case["batch"] - 1):
        rows.append(tuple(int(torch.randint(max(n // 2, k * d + 1), n + 1, (1,), generator=g))
                          for n, k, d in zip(size, kernel, dilation)))
    return rows


def _inputs(case, seed):
    size, kernel, dilation, _ = _params(case)
    dtype = getattr(torch, case["dtype"])
    B, H, Hkv, D = case["batch"], case["heads"], case["kv_heads"], case["dim"]
    g = torch.Generator(device="cuda").manual_seed(seed)

    def randn(*shape):
        return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).to(dtype)

    s = {}
    if case["op"] == "module":
        C = H * D
        s["x"] = randn(B, *size, C)
        for name, rows, cols in (("qkv", 3 * C, C), ("proj", C, C)):
            s[name + ".weight"] = randn(rows, cols) * cols ** -0.5
            s[name + ".bias"] = randn(rows) * 0.02
        s["do"] = randn(B, *size, C)
        return s
    if case["packed"]:
        qkv = randn(B, *size, 3, H, D)
        s["q"], s["k"], s["v"] = qkv.unbind(len(size) + 1)
    else:
        s["q"], s["k"], s["v"] = randn(B, *size, H, D), randn(B, *size, Hkv, D), randn(B, *size, Hkv, D)
    if case["op"] == "varlen":
        rows = _extents(case, seed)
        s["sizes"] = torch.tensor(rows if len(size) > 1 else [r[0] for r in rows], dtype=torch.int32)
    if case["op"] == "extra":
        s["gk"], s["gv"] = randn(B, case["tokens"], Hkv, D), randn(B, case["tokens"], Hkv, D)
    if case["op"] == "rpb":
        s["rpb"] = randn(H, *(2 * k - 1 for k in kernel))
    if case["grad"]:
        s["do"] = randn(B, *(-(-n // case["stride"]) for n in size), H, D)
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    size, kernel, dilation, causal = _params(case)
    rank = len(size)
    st = {"op": case["op"], "rank": rank, "do": s.get("do"), "grad": case["grad"], "scale": case["dim"] ** -0.5}
    if case["op"] == "module":
        cls = getattr(na, f"NeighborhoodAttention{rank}D")
        layer = cls(case["heads"] * case["dim"], case["heads"], kernel, dilation=dilation).to(
            device="cuda", dtype=getattr(torch, case["dtype"]))
        layer.load_state_dict({n: s[n] for n in ("qkv.weight", "qkv.bias", "proj.weight", "proj.bias")})
        st["layer"], st["x"] = layer, s["x"].requires_grad_(True)
        st["leaves"] = [st["x"], *layer.parameters()]
        return st
    names = [n for n in ("q", "k", "v", "gk", "gv", "rpb") if n in s]
    leaves = [s[n] for n in names]
    if case["grad"]:
        leaves = [t.detach().requires_grad_(True) for t in leaves]
    st["leaves"] = leaves
    st.update(zip(names, leaves))
    st["kw"] = dict(kernel_size=kernel, dilation=dilation)
    if case["op"] in ("na", "extra"):
        st["kw"].update(stride=case["stride"], is_causal=causal)
    if case["op"] == "varlen":
        st["sizes"] = s["sizes"]
    if case["op"] == "rpb":
        st["kw"] = dict(kernel_size=kernel[0], dilation=dilation[0])
    return st


def _forward(s):
    op, rank = s["op"], s["rank"]
    if op == "na":
        return getattr(na, f"na{rank}d")(s["q"], s["k"], s["v"], **s["kw"])
    if op == "extra":
        return getattr(na, f"na{rank}d")(s["q"], s["k"], s["v"], additional_keys=s["gk"], additional_values=s["gv"],
                                         **s["kw"])
    if op == "varlen":
        return getattr(na, f"na{rank}d_varlen")(s["q"], s["k"], s["v"], s["sizes"], **s["kw"])
    if op == "split":
        logits = getattr(na, f"na{rank}d_qk")(s["q"], s["k"], scale=s["scale"], **s["kw"])
        return getattr(na, f"na{rank}d_av")(logits.softmax(-1), s["v"], **s["kw"])
    if op == "rpb":
        logits = getattr(allin1, f"na{rank}d_qk_rpb")(s["q"], s["k"], s["rpb"], scale=s["scale"], **s["kw"])
        return getattr(allin1, f"na{rank}d_av_fused")(logits.softmax(-1), s["v"], **s["kw"])
    return s["layer"](s["x"])


def run(state):
    if not state["grad"]:
        with torch.no_grad():
            return _forward(state)
    out = _forward(state)
    return (out, *torch.autograd.grad(out, state["leaves"], state["do"]))


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------


def _axis_pairs(n, kernel, stride, causal, dilation):
    """Valid (query, key) pairs of one axis."""
    if not causal:
        return -(-n // stride) * kernel
    return sum(min(kernel, i // dilation + 1) for i in range(0, n, stride))


def work(case):
    size, kernel, dilation, causal = _params(case)
    esz = 4 if case["dtype"] == "float32" else 2
    B, H, Hkv, D = case["batch"], case["heads"], case["kv_heads"], case["dim"]
    n_in, n_out = math.prod(size), math.prod(-(-n // case["stride"]) for n in size)
    pairs = math.prod(_axis_pairs(n, k, case["stride"], c, d)
                      for n, k, d, c in zip(size, kernel, dilation, causal))
    pairs += n_out * case["tokens"]
    flops = (14.0 if case["grad"] else 4.0) * B * H * pairs * D
    q, o = B * n_in * H * D, B * n_out * H * D
    kv = 2 * B * (n_in + case["tokens"]) * Hkv * D
    elements = q + kv + o
    if case["grad"]:
        elements += o + q + kv
    if case["op"] in ("split", "rpb"):
        # logits, weights and the gradients of both pass between the calls:
        # each written once and read once
        elements += 8 * B * n_out * H * math.prod(kernel)
    if case["op"] == "rpb":
        elements += 2 * H * math.prod(2 * k - 1 for k in kernel)
    if case["op"] == "module":
        C = H * D
        # x and its gradient, y and its gradient, the parameters and theirs
        elements += 2 * 4 * (C * C + C)
        flops += 3 * 2.0 * B * n_in * C * 4 * C
    return {"bytes": float(esz * elements), "flops": flops}


def tolerance(case):
    # Seen against float64: 1e-7 to 4e-7 in single precision (a projection of
    # a few hundred channels adds as much again), 2e-3 to 2.5e-3 in bfloat16,
    # where probabilities and score gradients are rounded once before the
    # second product, and 6e-3 where logits, weights and their gradients pass
    # between calls in bfloat16.  float16 keeps three more bits.
    if case["dtype"] == "float32":
        return {"rel": 4e-6}
    rel = 2.4e-2 if case["op"] in ("split", "rpb", "module") else 1e-2
    return {"rel": rel / 8 if case["dtype"] == "float16" else rel}


# ---------------------------------------------------------------------------
# float64
# ---------------------------------------------------------------------------


def _axis_windows(n, kernel, dilation, stride, causal):
    """Key positions [n_out, K] of each query of one axis, and which are
    valid.  Queries attend within their residue class mod the dilation: class
    index c of a class of m members starts its window at c - K // 2, moved in
    at both ends; a causal window ends at the query."""
    pos = torch.arange(0, n, stride, device="cuda")
    cls, res = pos // dilation, pos % dilation
    if causal:
        first = cls - (kernel - 1)
    else:
        members = (n - res + dilation - 1) // dilation
        first = torch.minimum((cls - kernel // 2).clamp(min=0), members - kernel)
    member = first[:, None] + torch.arange(kernel, device="cuda")
    return member.clamp(min=0) * dilation + res[:, None], member >= 0


def _windows(size, kernel, dilation, stride, causal):
    """Flat key positions [n_queries, entries] and which are valid; and per
    entry and axis the key's class steps from its query, [n_queries, entries,
    rank]."""
    rank = len(size)
    flat = torch.zeros((1, 1), dtype=torch.long, device="cuda")
    ok = torch.ones((1, 1), dtype=torch.bool, device="cuda")
    steps = torch.zeros((1, 1, 0), dtype=torch.long, device="cuda")
    for a in range(rank):
        key, valid = _axis_windows(size[a], kernel[a], dilation[a], stride, causal[a])
        n, k = key.shape
        step = (key - torch.arange(0, size[a], stride, device="cuda")[:, None]) // dilation[a]
        m, e = flat.shape
        flat = (flat[:, None, :, None] * size[a] + key[None, :, None, :]).reshape(m * n, e * k)
        ok = (ok[:, None, :, None] & valid[None, :, None, :]).reshape(m * n, e * k)
        steps = torch.cat([steps[:, None, :, None, :].expand(m, n, e, k, a),
                           step[None, :, None, :, None].expand(m, n, e, k, 1)], dim=-1).reshape(m * n, e * k, a + 1)
    return flat, ok, steps


def _attend(q, k, v, do, flat, ok, scale, gk=None, gv=None, bias=None, bias_at=None):
    """Attention of q [B, N, H, D] over windows of k, v [B, M, Hkv, D], and
    with ``do`` its gradients (out, dq, dk, dv, dgk, dgv, dbias).  bias [H,
    T] is read at bias_at [N, entries]."""
    B, N, H, D = q.shape
    Hkv = k.shape[2]
    q = q.view(B, N, Hkv, H // Hkv, D)
    E, T = flat.shape[1], 0 if gk is None else gk.shape[1]
    logits = torch.empty(B, N, Hkv, H // Hkv, E + T, dtype=q.dtype, device=q.device)
    keys = [(lambda t, j=j: t[:, flat[:, j]].unsqueeze(3)) for j in range(E)]
    for j in range(E):
        logits[..., j] = (q * keys[j](k)).sum(-1) * scale
        if bias is not None:
            logits[..., j] += bias[:, bias_at[:, j]].t().view(1, N, Hkv, 1)
        logits[..., j].masked_fill_(~ok[:, j].view(1, N, 1, 1), -math.inf)
    for t in range(T):
        logits[..., E + t] = (q * gk[:, t, None, :, None]).sum(-1) * scale
    p = logits.softmax(-1)
    out = torch.zeros_like(q)
    for j in range(E):
        out += p[..., j, None] * keys[j](v)
    for t in range(T):
        out += p[..., E + t, None] * gv[:, t, None, :, None]
    if do is None:
        return (out.view(B, N, H, D),)
    do = do.view(B, N, Hkv, H // Hkv, D)
    delta = (do * out).sum(-1)
    dq, dk, dv = torch.zeros_like(q), torch.zeros_like(k), torch.zeros_like(v)
    dgk, dgv = (None, None) if gk is None else (torch.zeros_like(gk), torch.zeros_like(gv))
    dbias = None if bias is None else torch.zeros_like(bias)
    for j in range(E):
        ds = p[..., j] * ((do * keys[j](v)).sum(-1) - delta)
        dq += ds[..., None] * keys[j](k) * scale
        dk.index_add_(1, flat[:, j], (ds[..., None] * q).sum(3) * scale)
        dv.index_add_(1, flat[:, j], (p[..., j, None] * do).sum(3))
        if bias is not None:
            dbias.index_add_(1, bias_at[:, j], ds.sum(0).view(N, H).t().contiguous())
    for t in range(T):
        ds = p[..., E + t] * ((do * gv[:, t, None, :, None]).sum(-1) - delta)
        dq += ds[..., None] * gk[:, t, None, :, None] * scale
        dgk[:, t] = (ds[..., None] * q).sum((1, 3)) * scale
        dgv[:, t] = (p[..., E + t, None] * do).sum((1, 3))
    return out.view(B, N, H, D), dq.view(B, N, H, D), dk, dv, dgk, dgv, dbias


def exact(case, seed):
    s = {n: (t.double() if t.is_floating_point() else t) for n, t in _inputs(case, seed).items()}
    size, kernel, dilation, causal = _params(case)
    B, H, Hkv, D = case["batch"], case["heads"], case["kv_heads"], case["dim"]
    scale, st = D ** -0.5, case["stride"]
    n_out = tuple(-(-n // st) for n in size)
    if case["op"] == "module":
        C = H * D
        x = s["x"].reshape(-1, C)
        qkv = (x @ s["qkv.weight"].t() + s["qkv.bias"]).view(B, -1, 3, H, D)
        dy = s["do"].reshape(-1, C)
        do = (dy @ s["proj.weight"]).view(B, -1, H, D)
        flat, ok, _ = _windows(size, kernel, dilation, 1, causal)
        out, dq, dk, dv = _attend(*qkv.unbind(2), do, flat, ok, scale)[:4]
        out = out.reshape(-1, C)
        dqkv = torch.stack([dq, dk, dv], dim=2).reshape(-1, 3 * C)
        y = out @ s["proj.weight"].t() + s["proj.bias"]
        return (y.view_as(s["x"]), (dqkv @ s["qkv.weight"]).view_as(s["x"]), dqkv.t() @ x, dqkv.sum(0), dy.t() @ out,
                dy.sum(0))
    if case["op"] == "varlen":
        got = [torch.zeros_like(s["q"]) for _ in range(4)]
        for b, ext in enumerate(_extents(case, seed)):
            at = (slice(b, b + 1), *(slice(0, n) for n in ext))
            part = [s[n][at].reshape(1, -1, H, D) for n in ("q", "k", "v", "do")]
            flat, ok, _ = _windows(ext, kernel, dilation, 1, causal)
            for whole, r in zip(got, _attend(*part, flat, ok, scale)):
                whole[at] = r.view(1, *ext, H, D)
        return tuple(got)
    flat, ok, steps = _windows(size, kernel, dilation, st, causal)
    at = (slice(None), *(slice(0, None, st) for _ in size))
    do = s["do"].reshape(B, -1, H, D) if case["grad"] else None
    bias = bias_at = None
    if case["op"] == "rpb":
        bias = s["rpb"].reshape(H, -1)
        bias_at = torch.zeros_like(flat)
        for a, k in enumerate(kernel):
            bias_at = bias_at * (2 * k - 1) + steps[..., a] + k - 1
    got = _attend(s["q"][at].reshape(B, -1, H, D), s["k"].reshape(B, -1, Hkv, D), s["v"].reshape(B, -1, Hkv, D), do,
                  flat, ok, scale, s.get("gk"), s.get("gv"), bias, bias_at)
    out = got[0].view(B, *n_out, H, D)
    if not case["grad"]:
        return out
    dq = torch.zeros_like(s["q"])
    dq[at] = got[1].view(B, *n_out, H, D)
    res = (out, dq, got[2].view_as(s["k"]), got[3].view_as(s["v"]))
    if case["op"] == "extra":
        res += (got[4], got[5])
    if case["op"] == "rpb":
        res += (got[6].view_as(s["rpb"]),)
    return res
