"""Variable-length and global-key calls through the C++ binding: a repeated
signature gives the first call's bits, and sample extents reach the device
whatever their number."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.fixture(autouse=True)
def _hip():
    import natten_mps_amd

    natten_mps_amd.set_backend("hip")
    yield


@pytest.mark.parametrize("rank", [1, 2, 3])
@pytest.mark.parametrize("batch", [1, 256, 257, 600])  # 256 samples per launch
@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_varlen_extents_reach_the_device(rank, batch, dtype):
    from natten_mps_amd._core import hip

    g = torch.Generator().manual_seed(batch + rank)
    sizes = torch.randint(3, 1 << 20, (batch, rank), generator=g, dtype=dtype)
    want = torch.cat([torch.ones(batch, 3 - rank, dtype=torch.int32), sizes.to(torch.int32)], dim=1)
    got = hip.varlen_extents(rank, sizes, DEV)
    assert got.dtype == torch.int32 and torch.equal(got.cpu(), want)
    assert hip.varlen_extents(rank, got, DEV) is got
    assert torch.equal(hip.varlen_extents(rank, sizes.to(DEV), DEV).cpu(), want)


def _step(kind, leaves, do):
    from natten_mps_amd import functional as F

    if kind == "varlen":
        out = F.na2d_varlen(*leaves, torch.tensor([[12, 20], [17, 11]]), kernel_size=(5, 7))
    else:
        out = F.na2d(*leaves[:3], kernel_size=(5, 7), additional_keys=leaves[3], additional_values=leaves[4])
    return [t.detach().clone() for t in (out, *torch.autograd.grad(out, leaves, do))]


@pytest.mark.parametrize("kind", ["varlen", "global"])
def test_repeated_calls_give_the_first_calls_bits(kind):
    """The first call registers the signature, later ones run it in C++, also
    on another stream and with new inputs in between."""
    from natten_mps_amd._core import _lib

    _lib.binding().clear()
    g = torch.Generator().manual_seed(5)
    shapes = [(2, 17, 20, 2, 32)] * 3 + ([(2, 9, 2, 32)] * 2 if kind == "global" else [])
    make = lambda: [torch.randn(s, generator=g).to(torch.bfloat16).to(DEV).requires_grad_(True) for s in shapes]  # noqa: E731
    leaves, other = make(), make()
    do = torch.randn(shapes[0], generator=g).to(torch.bfloat16).to(DEV)
    first = _step(kind, leaves, do)
    changed = _step(kind, other, do)
    assert not torch.equal(first[0], changed[0])
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        second = _step(kind, leaves, do)
    torch.cuda.current_stream().wait_stream(side)
    for a, b in zip(first, second):
        assert torch.equal(a, b)


def test_unused_lse_brings_no_gradient():
    """out alone, lse alone and both: the gradients add up as autograd's do."""
    from natten_mps_amd import functional as F

    g = torch.Generator().manual_seed(6)
    leaves = [torch.randn(1, 15, 16, 2, 32, generator=g).to(DEV).requires_grad_(True) for _ in range(3)]
    do, dl = torch.randn(1, 15, 16, 2, 32, generator=g).to(DEV), torch.randn(1, 15, 16, 2, generator=g).to(DEV)

    def grads(use_out, use_lse):
        out, lse = F.na2d(*leaves, kernel_size=5, return_lse=True)
        return torch.autograd.grad([t for t, u in ((out, use_out), (lse, use_lse)) if u], leaves,
                                   [t for t, u in ((do, use_out), (dl, use_lse)) if u], allow_unused=True)

    both, a, b = grads(True, True), grads(True, False), grads(False, True)
    for x, y, z in zip(both, a, b):
        s = y if z is None else y + z
        torch.testing.assert_close(x, s, atol=2e-5, rtol=2e-5)
