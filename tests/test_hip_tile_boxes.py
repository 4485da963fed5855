"""Query tiles of 8 rows by 4 columns (csrc/na_mfma.hip): in-plane kernels of
up to 5 columns, at sizes where the boxes end ragged or the rule just applies,
against the CPU oracle."""

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
    # spatial, heads q / kv, dim, kernel, dilation, causal
    ((3, 8, 8), 1, 1, 64, (3, 5, 5), (1, 1, 1), (False, False, False)),     # the smallest
    ((5, 9, 13), 2, 2, 32, (3, 3, 5), (1, 1, 1), (False, False, False)),
    ((6, 17, 22), 4, 2, 128, (3, 5, 4), (2, 2, 2), (False, True, False)),
    ((4, 10, 15), 2, 2, 96, (1, 5, 5), (1, 1, 1), (False, False, True)),    # no depth window
    ((7, 16, 12), 2, 2, 32, (5, 7, 2), (1, 1, 1), (True, False, False)),
    ((19, 30), 2, 1, 128, (5, 5), (1, 1), (False, False)),
    ((33, 9), 2, 2, 96, (7, 3), (1, 1), (False, True)),
    ((5, 8, 16), 2, 2, 32, (3, 7, 7), (1, 1, 1), (False, False, False)),    # one plane of 8 x 8 at head dim 32
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", CASES)
def test_narrow_query_tiles_match_oracle(case, dtype):
    from natten_mps_amd import functional as F
    from natten_mps_amd._core import _lib

    sp, hq, hkv, dim, ks, dil, causal = case
    rank = len(sp)
    print(case, dtype, flush=True)
    g = torch.Generator().manual_seed(51)
    q, k, v, do = (torch.randn(2, *sp, h, dim, generator=g).to(dtype) for h in (hq, hkv, hkv, hq))
    dl = torch.randn(2, *sp, hq, generator=g)
    leaves = [t.to(DEV).requires_grad_(True) for t in (q, k, v)]
    _lib.profile_read(reset=True)
    _lib.profile_enable(True)
    try:
        out, lse = getattr(F, f"na{rank}d")(*leaves, kernel_size=ks, dilation=dil, is_causal=causal, return_lse=True)
        grads = torch.autograd.grad((out, lse), leaves, (do.to(DEV), dl.to(DEV)))
        torch.cuda.synchronize()
    finally:
        _lib.profile_enable(False)
    launched = set(_lib.profile_read(reset=True))
    assert {"na_fwd_mfma", "na_bwd_q_mfma"} <= launched, launched
    rq, rk, rv = (t.float().requires_grad_(True) for t in (q, k, v))
    ke, ve = (t.repeat_interleave(hq // hkv, dim=-2) for t in (rk, rv))
    st = (1,) * rank
    logits = getattr(P, f"na{rank}d_qk_forward")(rq, ke, ks, dil, st, causal, dim ** -0.5)
    ref = getattr(P, f"na{rank}d_av_forward")(torch.softmax(logits, dim=-1), ve, ks, dil, st, causal)
    ref_lse = torch.logsumexp(logits, dim=-1)
    rgrads = torch.autograd.grad((ref, ref_lse), (rq, rk, rv), (do.float(), dl))
    for name, a, b in zip(("out", "lse", "dq", "dk", "dv"), (out, lse, *grads), (ref, ref_lse, *rgrads)):
        assert_parity(a.detach().cpu(), b.detach(), dtype, name)
