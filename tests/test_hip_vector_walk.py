"""The vector kernels' pipelined walks (csrc/na_generic.hip): head dims that
leave lanes idle or give a lane two pieces of a row, group counts from 8 down
to 1, ragged row ends, windows clipped on either side, against the oracle in
float64."""

import pytest
import torch

import oracle.pure as P
from _parity import assert_parity

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.fixture(autouse=True)
def _hip():
    import natten_mps_amd

    natten_mps_amd.set_backend("hip")
    yield


CASES = [
    # spatial, batch, heads q / kv, dim, kernel, dilation, causal
    ((11, 14), 1, 2, 2, 24, (5, 6), (1, 1), (False, False)),     # 8 groups of few lanes
    ((19, 23), 2, 4, 2, 40, (3, 7), (2, 3), (False, True)),      # GQA
    ((33, 29), 2, 2, 2, 72, (11, 10), (1, 1), (False, False)),
    ((12, 12), 1, 1, 1, 136, (3, 3), (1, 4), (True, False)),     # 16 dims a lane
    ((70, 70), 8, 4, 4, 16, (3, 3), (1, 1), (False, False)),     # one group a query
    ((97,), 2, 2, 2, 56, (13,), (2,), (True,)),
    ((128,), 1, 2, 1, 8, (33,), (3,), (False,)),
    ((5, 9, 8), 1, 2, 2, 48, (3, 4, 5), (1, 2, 1), (False, False, True)),
]


def _case(case, dtype, seed=41):
    sp, b, hq, hkv, dim, ks, dil, causal = case
    print(case, dtype, flush=True)
    g = torch.Generator().manual_seed(seed)
    r = lambda h: torch.randn(b, *sp, h, dim, generator=g).to(dtype)  # noqa: E731
    q, k, v, do = r(hq), r(hkv), r(hkv), r(hq)
    rank = len(sp)
    ref = [t.double().requires_grad_(True) for t in (q, k, v)]
    args = (ks, dil, (1,) * rank, causal)
    dev = [t.to(DEV).requires_grad_(True) for t in (q, k, v)]
    return rank, dev, ref, do, args


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("case", CASES)
def test_fused(case, dtype):
    from natten_mps_amd import functional as F

    rank, dev, ref, do, (ks, dil, st, causal) = _case(case, dtype)
    out, lse = getattr(F, f"na{rank}d")(*dev, kernel_size=ks, dilation=dil, is_causal=causal, return_lse=True)
    grads = torch.autograd.grad(out, dev, do.to(DEV))
    n = dev[0].shape[-2] // dev[1].shape[-2]
    k, v = (t.repeat_interleave(n, dim=-2) for t in ref[1:])
    logits = getattr(P, f"na{rank}d_qk_forward")(ref[0], k, ks, dil, st, causal, case[4] ** -0.5)
    want = getattr(P, f"na{rank}d_av_forward")(torch.softmax(logits, dim=-1), v, ks, dil, st, causal)
    rgrads = torch.autograd.grad(want, ref, do.double())
    for name, a, b in zip(("out", "lse", "dq", "dk", "dv"), (out, lse, *grads),
                          (want, torch.logsumexp(logits, dim=-1), *rgrads)):
        assert_parity(a.detach().cpu(), b.detach(), dtype, name)


@pytest.mark.parametrize("case", [c for c in CASES if c[2] == c[3]])
def test_split(case):
    """fp32 operands: logits and their gradients within 8 ulp of a dot
    product's largest partial sum, gathers (64-bit sums) within 2 ulp."""
    from natten_mps_amd import functional as F

    rank, (q, k, v), (rq, rk, rv), do, (ks, dil, st, causal) = _case(case, torch.float32)
    kw = dict(kernel_size=ks, dilation=dil, is_causal=causal)
    logits = getattr(F, f"na{rank}d_qk")(q, k, **kw)
    ref = getattr(P, f"na{rank}d_qk_forward")(rq, rk, ks, dil, st, causal, None)
    ok = torch.isfinite(ref)
    assert torch.equal(torch.isfinite(logits).cpu(), ok)
    eps = torch.finfo(torch.float32).eps
    big = float(rq.detach().abs().amax() * rk.detach().abs().amax()) * case[4]
    assert float((logits.detach().cpu().double() - ref.detach())[ok].abs().max()) <= 8 * eps * big
    w = torch.softmax(ref, dim=-1).detach().float()
    a = w.to(DEV).requires_grad_(True)
    out = getattr(F, f"na{rank}d_av")(a, v, **kw)
    da, dv = torch.autograd.grad(out, (a, v), do.to(DEV))
    rw = w.double().requires_grad_(True)
    want = getattr(P, f"na{rank}d_av_forward")(rw, rv, ks, dil, st, causal)
    rda, rdv = torch.autograd.grad(want, (rw, rv), do.double())
    g = torch.where(ok, torch.randn(ref.shape, generator=torch.Generator().manual_seed(7)), torch.zeros(()))
    dq, dk = torch.autograd.grad(logits, (q, k), g.to(DEV))
    rdq, rdk = torch.autograd.grad(ref, (rq, rk), torch.where(ok, g.double(), torch.zeros((), dtype=torch.float64)))
    for name, x, y in (("out", out, want), ("dv", dv, rdv), ("dq", dq, rdq), ("dk", dk, rdk)):
        x, y = x.detach().cpu().double(), y.detach()
        assert bool(((x - y).abs() <= 2 * eps * y.abs() + 1e-12).all()), (name, float((x - y).abs().max()))
    diff = (da.detach().cpu().double() - rda)[ok].abs().max()
    assert float(diff) <= 8 * eps * float(do.abs().amax() * rv.detach().abs().amax()) * case[4]
