"""The band kernels (csrc/na_band.hip): in-plane windows of 10 to 16 columns,
staged a band of union rows at a time.  Sizes at the edges of their tiles
(128 items in rows of 8 or 16 columns; bands of 2 or 4 rows), on every head
dim, against the CPU oracle."""

import pytest
import torch

import oracle.pure as P
from _parity import assert_parity

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.fixture(autouse=True)
def _hip(monkeypatch):
    import natten_mps_amd

    natten_mps_amd.set_backend("hip")
    # small grids run on the general tiles where those hold the problem
    monkeypatch.setenv("NATTEN_HIP_BAND", "1")
    yield


CASES = [
    # spatial, heads q / kv, dim, kernel, dilation, causal, packed
    ((17, 33), 2, 2, 64, (13, 13), (1, 1), (False, False), False),
    ((16, 13), 1, 1, 32, (3, 13), (1, 1), (False, False), False),   # one column of windows
    ((8, 40), 2, 2, 64, (1, 11), (1, 1), (False, False), False),    # no window rows to walk
    ((29, 45), 2, 2, 32, (13, 13), (1, 1), (True, False), False),
    ((23, 44), 4, 2, 64, (7, 11), (1, 1), (False, True), False),    # GQA
    ((50, 31), 2, 2, 128, (15, 15), (2, 2), (False, False), False),
    ((21, 36), 2, 1, 128, (5, 16), (1, 2), (False, False), False),  # even kernel
    ((40, 20), 2, 2, 64, (33, 10), (1, 1), (False, False), True),   # packed q/k/v views
    ((27, 49), 3, 3, 32, (11, 11), (2, 3), (True, True), True),
]


def _inputs(seed, shapes, dtype):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn(s, generator=g, dtype=torch.float32).to(dtype) for s in shapes]


# Windows whose query side stays on the 8 x 8 tiles: the key tiles at the
# border, or of classes about twice the kernel, do not fit those.
KEY_SIDE_CASES = [
    ((40, 64), 2, 2, 64, (9, 9), (1, 1), (False, False), False),
    ((40, 32), 2, 2, 32, (8, 8), (1, 1), (False, False), False),
    ((22, 22), 2, 2, 32, (7, 7), (1, 1), (False, False), True),
    ((48, 48), 2, 1, 32, (9, 9), (2, 2), (False, False), False),
]
# Head dim 128 takes both sides from 8 columns; so does a backward whose key
# side no other tile kernel holds.
WIDE_CASES = [((21, 37), 2, 1, 128, (9, 9), (1, 1), (True, False), False),
              ((19, 40), 1, 1, 128, (5, 8), (1, 2), (False, False), True)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", CASES + WIDE_CASES)
def test_band_kernels_match_oracle(case, dtype):
    _check(case, dtype, {"na_fwd_band", "na_bwd_q_band", "na_bwd_kv_band"})


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", KEY_SIDE_CASES)
def test_band_key_side_matches_oracle(case, dtype):
    assert not any("q_band" in n for n in _check(case, dtype, {"na_bwd_kv_band"}))


def _check(case, dtype, names):
    """Output, log-sum-exp and the gradients through both."""
    from natten_mps_amd import functional as F
    from natten_mps_amd._core import _lib

    sp, hq, hkv, dim, ks, dil, causal, packed = case
    print(case, dtype, flush=True)
    q, k, v, do = _inputs(31, [(2, *sp, hq, dim), (2, *sp, hkv, dim), (2, *sp, hkv, dim), (2, *sp, hq, dim)], dtype)
    (dl,) = _inputs(32, [(2, *sp, hq)], dtype)
    dev = [t.to(DEV) for t in (q, k, v)]
    if packed:
        dev = list(torch.stack(dev, dim=3).unbind(3))
    leaves = [t.requires_grad_(True) for t in dev]
    _lib.profile_read(reset=True)
    _lib.profile_enable(True)
    try:
        out, lse = F.na2d(*leaves, kernel_size=ks, dilation=dil, is_causal=causal, return_lse=True)
        grads = torch.autograd.grad((out, lse), leaves, (do.to(DEV), dl.to(DEV)))
        torch.cuda.synchronize()
    finally:
        _lib.profile_enable(False)
    launched = set(_lib.profile_read(reset=True))
    assert names <= launched, launched

    rq, rk, rv = (t.float().requires_grad_(True) for t in (q, k, v))
    n = hq // hkv
    ke, ve = (t.repeat_interleave(n, dim=-2) for t in (rk, rv))
    logits = P.na2d_qk_forward(rq, ke, ks, dil, (1, 1), causal, dim ** -0.5)
    ref_lse = torch.logsumexp(logits, dim=-1)
    ref = P.na2d_av_forward(torch.softmax(logits, dim=-1), ve, ks, dil, (1, 1), causal)
    rgrads = torch.autograd.grad((ref, ref_lse), (rq, rk, rv), (do.float(), dl.float()))
    for name, a, b in zip(("out", "lse", "dq", "dk", "dv"), (out, lse, *grads), (ref, ref_lse, *rgrads)):
        assert_parity(a.detach().cpu(), b.detach(), dtype, name)
    return launched


# Calls whose alternative is the vector kernels (fp32 probabilities).
TWO_TERM_CASES = [((24, 40), 64, (13, 13)), ((17, 30), 64, (9, 9)), ((24, 33), 128, (13, 15)),
                  ((30, 21), 128, (9, 9)), ((80, 20), 32, (33, 13))]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", TWO_TERM_CASES)
def test_two_term_products_add_no_error(case, dtype):
    """The gradients' error against float64 is that of rounding them once
    (one-term probabilities, rounded as often as the result, add to that; two
    terms leave 2^-17, a 256th of one rounding)."""
    from natten_mps_amd import functional as F
    from natten_mps_amd._core import _lib

    sp, dim, ks = case
    print(case, dtype, flush=True)
    ts = _inputs(35, [(2, *sp, 2, dim)] * 4, dtype)
    leaves = [t.to(DEV).requires_grad_(True) for t in ts[:3]]
    _lib.profile_read(reset=True)
    _lib.profile_enable(True)
    try:
        out = F.na2d(*leaves, kernel_size=ks)
        grads = torch.autograd.grad(out, leaves, ts[3].to(DEV))
        torch.cuda.synchronize()
    finally:
        _lib.profile_enable(False)
    assert {"na_bwd_q_band", "na_bwd_kv_band"} <= set(_lib.profile_read(reset=True))
    q, k, v = (t.double().requires_grad_(True) for t in ts[:3])
    one = (1, 1)
    w = torch.softmax(P.na2d_qk_forward(q, k, ks, one, one, (False, False), dim ** -0.5), dim=-1)
    ref = P.na2d_av_forward(w, v, ks, one, one, (False, False))
    rgrads = torch.autograd.grad(ref, (q, k, v), ts[3].double())
    for name, a, b in zip(("dq", "dk", "dv"), grads, rgrads):
        b = b.detach()
        err = float((a.cpu().double() - b).norm())
        assert err <= 1.03 * float((b.to(dtype).double() - b).norm()), (name, err)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("scales", [(1e-2, 1), (1e-3, 1), (1e-4, 1), (1e-3, 4), (100, 1)])  # of dO and k
@pytest.mark.parametrize("case", [TWO_TERM_CASES[2], TWO_TERM_CASES[4], ((200, 19), 32, (97, 16))])
def test_two_term_products_keep_small_gradients(case, scales, dtype):
    """The bound of test_two_term_products_add_no_error where dS or P leaves
    the range in which two unscaled fp16 terms hold it: a mean-reduced loss's
    gradients, and windows of hundreds of keys.  (The forward takes two terms
    in these cases: a one-term forward's log-sum-exp adds 4 % at 4 k.)"""
    from natten_mps_amd import functional as F

    sp, dim, ks = case
    print(case, scales, dtype, flush=True)
    q, k, v, do = _inputs(35, [(1, *sp, 2, dim)] * 4, torch.float32)
    ts = [t.to(dtype) for t in (q, k * scales[1], v, do * scales[0])]
    leaves = [t.to(DEV).requires_grad_(True) for t in ts[:3]]
    out = F.na2d(*leaves, kernel_size=ks)
    grads = torch.autograd.grad(out, leaves, ts[3].to(DEV))
    one, no = (1, 1), (False, False)
    q, k, v = (t.double().requires_grad_(True) for t in ts[:3])
    logits = P.na2d_qk_forward(q, k, ks, one, one, no, dim ** -0.5)
    ref = P.na2d_av_forward(torch.softmax(logits, dim=-1), v, ks, one, one, no)
    rgrads = torch.autograd.grad(ref, (q, k, v), ts[3].double())
    for name, a, b in zip(("dq", "dk", "dv"), grads, rgrads):
        b = b.detach()
        err = float((a.cpu().double() - b).norm())
        assert err <= 1.03 * float((b.to(dtype).double() - b).norm()), (name, err)


@pytest.mark.parametrize("tokens", [1, 7])
@pytest.mark.parametrize("ks", [(9, 9), (7, 7)])  # key side on the band and on the lean tiles
def test_window_key_side_under_global_keys(ks, tokens):
    """dK / dV of the window with global keys beside it."""
    from natten_mps_amd import functional as F

    shapes = [(2, 33, 40, 2, 64)] * 3 + [(2, tokens, 2, 64)] * 2 + [(2, 33, 40, 2, 64)]
    *ts, do = _inputs(34, shapes, torch.bfloat16)
    leaves = [t.to(DEV).requires_grad_(True) for t in ts]
    out = F.na2d(*leaves[:3], kernel_size=ks, additional_keys=leaves[3], additional_values=leaves[4])
    grads = torch.autograd.grad(out, leaves, do.to(DEV))
    q, k, v, gk, gv = (t.float().requires_grad_(True) for t in ts)
    one = (1, 1)
    logits = P.na2d_qk_forward(q, k, ks, one, one, (False, False), 64 ** -0.5)
    extra = torch.einsum("bxyhd,bthd->bxyht", q, gk) * 64 ** -0.5
    w = torch.softmax(torch.cat([logits, extra], dim=-1), dim=-1)
    n = logits.shape[-1]
    ref = P.na2d_av_forward(w[..., :n], v, ks, one, one, (False, False)) + torch.einsum(
        "bxyht,bthd->bxyhd", w[..., n:], gv)
    rgrads = torch.autograd.grad(ref, (q, k, v, gk, gv), do.float())
    for name, a, b in zip(("out", "dq", "dk", "dv", "dgk", "dgv"), (out, *grads), (ref, *rgrads)):
        assert_parity(a.detach().cpu(), b.detach(), torch.bfloat16, name)


def test_band_kernels_recompute_non_finite_operands():
    """A non-finite key outside a query's window does not reach it, and one
    inside does, as in the oracle (the finite elements agree)."""
    from natten_mps_amd import functional as F

    ks = (13, 13)
    q, k, v, do = _inputs(33, [(1, 20, 34, 1, 64)] * 4, torch.bfloat16)
    k[0, 3, 5, 0, 7] = float("inf")
    v[0, 15, 30, 0, 9] = float("nan")
    leaves = [t.to(DEV).requires_grad_(True) for t in (q, k, v)]
    out = F.na2d(*leaves, kernel_size=ks)
    grads = torch.autograd.grad(out, leaves, do.to(DEV))
    ref_leaves = [t.float().requires_grad_(True) for t in (q, k, v)]
    ref = P.na2d_forward(*ref_leaves, ks, (1, 1), (1, 1), (False, False), None)
    rgrads = torch.autograd.grad(ref, ref_leaves, do.float())
    for name, a, b in zip(("out", "dq", "dk", "dv"), (out, *grads), (ref, *rgrads)):
        a, b = a.detach().float().cpu(), b.detach()
        assert torch.equal(torch.isfinite(a), torch.isfinite(b)), name
        fin = torch.isfinite(b)
        assert_parity(a[fin], b[fin], torch.bfloat16, name)


# batch, spatial, heads, dim, kernel, dilation, and which of the forward, dQ
# and dK/dV run on the band kernels by themselves
ROUTE_CASES = [
    (1, (20, 20), 1, 64, (3, 13), (1, 1), ""),          # a few workgroups
    (4, (56, 56), 8, 64, (11, 11), (4, 4), ""),         # classes of 14: 64-query tiles in 64 KB
    (4, (128, 128), 8, 64, (3, 13), (1, 1), "fq"),      # 32-query tiles
    (8, (64, 64), 8, 32, (9, 9), (1, 1), "k"),          # key tiles of 16
    (4, (64, 64), 8, 64, (8, 8), (1, 1), "k"),          # key tiles past 64 KB
    (1, (64, 64), 1, 64, (9, 9), (1, 1), ""),           # the same, one image of one head
    (2, (64, 64), 4, 64, (5, 11), (1, 1), "fqk"),       # past 64 KB, or 16-query tiles
    (8, (28, 28), 8, 128, (8, 8), (2, 2), "fk"),        # dQ: its registers leave one workgroup per CU
]


@pytest.mark.parametrize("case", ROUTE_CASES)
def test_each_side_takes_the_faster_kernels(case, monkeypatch):
    """The route that the sizes give, and both routes' results beside each
    other (bfloat16, probabilities rounded once on either)."""
    from natten_mps_amd import functional as F
    from natten_mps_amd._core import _lib

    B, sp, heads, dim, ks, dil, want = case
    print(case, flush=True)
    g = torch.Generator(device=DEV).manual_seed(41)
    ts = [torch.randn(B, *sp, heads, dim, generator=g, device=DEV).bfloat16() for _ in range(4)]
    leaves = [t.requires_grad_(True) for t in ts[:3]]

    def run():
        _lib.profile_read(reset=True)
        _lib.profile_enable(True)
        try:
            out = F.na2d(*leaves, kernel_size=ks, dilation=dil)
            res = (out.detach(), *torch.autograd.grad(out, leaves, ts[3]))
            torch.cuda.synchronize()
        finally:
            _lib.profile_enable(False)
        names = {"na_fwd_band": "f", "na_bwd_q_band": "q", "na_bwd_kv_band": "k"}
        launched = _lib.profile_read(reset=True)
        return res, "".join(v for n, v in names.items() if n in launched)

    monkeypatch.setenv("NATTEN_HIP_BAND", "0")
    general, none = run()
    monkeypatch.delenv("NATTEN_HIP_BAND")
    chosen, got = run()
    assert none == "" and got == want, (none, got)
    for name, a, b in zip(("out", "dq", "dk", "dv"), chosen, general):
        assert_parity(a.cpu(), b.cpu().float(), torch.bfloat16, name)
