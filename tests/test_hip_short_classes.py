"""Key tiles of classes about two kernels long on the 8 x 8 tile kernels
(csrc/na_lean.hip): both borders meet in one wave, whose keys are then attended
from the whole class -- 13 or 14 rows at a 7-row window, 7 chunks of a 1-D tile
at a window of 97.  Only the widest key-side instance holds them, so a launch
of the tiles' key side at these sizes is that instance's."""

import pytest
import torch

import oracle.pure as P
from _parity import assert_parity

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")

CASES = [
    # spatial, heads q / kv, dim, kernel, dilation, causal
    ((13, 14), 2, 2, 32, (7, 7), (1, 1), (False, False)),
    ((14, 14), 4, 2, 64, (7, 7), (1, 1), (False, False)),   # GQA
    ((28, 28), 2, 2, 64, (7, 7), (2, 2), (False, False)),   # (weight rows of one head would have an odd stride)
    ((14, 14), 2, 2, 32, (7, 7), (1, 1), (False, False)),
    ((14, 30), 2, 2, 32, (7, 5), (1, 1), (False, True)),
    ((200,), 2, 2, 64, (97,), (1,), (False,)),              # 1-D
    ((203,), 2, 1, 32, (97,), (1,), (False,)),
]
SPLIT_CASES = [c for c in CASES if len(c[0]) == 2 and c[1] == c[2] and not any(c[6])]
DTYPES = [torch.bfloat16, torch.float16, torch.float32]


@pytest.fixture(autouse=True)
def _hip():
    import natten_mps_amd

    natten_mps_amd.set_backend("hip")
    yield


def _inputs(case, dtype):
    sp, hq, hkv, dim = case[:4]
    print(case, dtype, flush=True)
    g = torch.Generator().manual_seed(61)
    return [torch.randn(2, *sp, h, dim, generator=g).to(dtype) for h in (hq, hkv, hkv, hq)]


def _launched(fn):
    from natten_mps_amd._core import _lib

    _lib.profile_read(reset=True)
    _lib.profile_enable(True)
    try:
        res = fn()
        torch.cuda.synchronize()
    finally:
        _lib.profile_enable(False)
    return res, set(_lib.profile_read(reset=True))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("case", CASES)
def test_fused_backward(case, dtype):
    from natten_mps_amd import functional as F

    sp, hq, hkv, dim, ks, dil, causal = case
    rank = len(sp)
    q, k, v, do = _inputs(case, dtype)
    leaves = [t.to(DEV).requires_grad_(True) for t in (q, k, v)]

    def step():
        out = getattr(F, f"na{rank}d")(*leaves, kernel_size=ks, dilation=dil, is_causal=causal)
        return (out, *torch.autograd.grad(out, leaves, do.to(DEV)))

    got, launched = _launched(step)
    assert "na_bwd_kv_lean" in launched, launched
    # windows of up to 97 keys: fp32 against float64 (see _parity)
    ref_dtype = torch.float64 if dtype == torch.float32 else torch.float32
    rq, rk, rv = (t.to(ref_dtype).requires_grad_(True) for t in (q, k, v))
    ke, ve = (t.repeat_interleave(hq // hkv, dim=-2) for t in (rk, rv))
    ref = getattr(P, f"na{rank}d_forward")(rq, ke, ve, ks, (1,) * rank, dil, causal, None)
    rgrads = torch.autograd.grad(ref, (rq, rk, rv), do.to(ref_dtype))
    for name, a, b in zip(("out", "dq", "dk", "dv"), got, (ref, *rgrads)):
        assert_parity(a.detach().cpu(), b.detach(), dtype, name)


@pytest.mark.parametrize("dtype", DTYPES[:2])
@pytest.mark.parametrize("case", SPLIT_CASES)
def test_split_backward(case, dtype):
    from natten_mps_amd import functional as F

    sp, _, _, dim, ks, dil, _ = case
    q, k, v, do = _inputs(case, dtype)
    leaves = [t.to(DEV).requires_grad_(True) for t in (q, k, v)]

    def step():
        w = F.na2d_qk(leaves[0], leaves[1], kernel_size=ks, dilation=dil, scale=dim ** -0.5).softmax(-1)
        out = F.na2d_av(w, leaves[2], kernel_size=ks, dilation=dil)
        return (out, *torch.autograd.grad(out, leaves, do.to(DEV)))

    got, launched = _launched(step)
    assert {"na_qk_bwd_k_lean", "na_av_bwd_v_lean"} <= launched, launched
    rq, rk, rv = (t.float().requires_grad_(True) for t in (q, k, v))
    ref = P.na2d_forward(rq, rk, rv, ks, (1, 1), dil, (False, False), None)
    rgrads = torch.autograd.grad(ref, (rq, rk, rv), do.float())
    for name, a, b in zip(("out", "dq", "dk", "dv"), got, (ref, *rgrads)):
        assert_parity(a.detach().cpu(), b.detach(), dtype, name)
