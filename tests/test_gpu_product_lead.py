"""GPU tests of how far ahead the gradient products load, against fp64: dHidden on both sides of the rule, by the length of its
contraction, in whole tiles and in pieces, with tokens that carry no gradient; both products of the recomputing backward."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture
def whole_tiles(request):
    """dHidden without a division of its contraction (as at token counts of whole device rounds), or with its own plan."""
    from fgrpo import _lib
    before = _lib.get_tuning("tail_split")
    _lib.set_tuning(tail_split=0 if request.param else before)
    yield request.param
    _lib.set_tuning(tail_split=before)


@pytest.mark.parametrize("whole_tiles", [True, False], indirect=True)
@pytest.mark.parametrize("T,H,V", [(60, 320, 59900), (700, 320, 59900), (60, 320, 60001), (257, 320, 60001), (700, 1088, 60001),
                                   (700, 1088, 59900), (2100, 320, 120100)])
def test_dhidden_on_both_sides_of_its_lead(dev, whole_tiles, T, H, V):
    """A kept numerator, the weight and the stored gradient are bf16: 2^-9 each of the norm at most, 6e-3 together."""
    from fgrpo import ops
    g = torch.Generator(device=dev).manual_seed(T + V)
    h = torch.randn(T, H, generator=g, device=dev).bfloat16().requires_grad_(True)
    w = (torch.randn(V, H, generator=g, device=dev) * (2.0 / H) ** 0.5).bfloat16().requires_grad_(True)
    y = torch.randint(0, V, (T,), generator=g, device=dev)
    up = torch.randn(T, generator=g, device=dev) / T
    up[20:50] = 0.0
    up[256:600] = 0.0                          # a row tile without any, and part of the next
    assert ops.keep_supported(T, H, V, torch.bfloat16)
    lp, _ = ops.lmhead_logprob(h, w, None, y, keep_logits="whole")
    dh, dw = torch.autograd.grad(lp, (h, w), up)
    hd, wd = h.detach().double(), w.detach().double()
    ds = -torch.softmax(hd @ wd.t(), 1)
    ds[torch.arange(T, device=dev), y] += 1
    ds *= up[:, None].double()
    for got, want in ((dh, ds @ wd), (dw, ds.t() @ hd)):
        assert (got.double() - want).norm() <= 6e-3 * want.norm() + 1e-12
    assert not dh[20:50].any()


@pytest.mark.parametrize("T,H", [(1, 320), (60, 320), (64, 1088), (65, 1088), (300, 320), (700, 1088), (2100, 320)])
def test_gradients_of_the_recomputing_backward(dev, T, H):
    """dLogits, the weight (dH) or the hidden row (dW) and the stored gradient are bf16: 2^-9 each, 6e-3 together."""
    from fgrpo import ops
    V = 33001
    g = torch.Generator(device=dev).manual_seed(T + H)
    h = torch.randn(T, H, generator=g, device=dev).bfloat16().requires_grad_(True)
    w = (torch.randn(V, H, generator=g, device=dev) * (2.0 / H) ** 0.5).bfloat16().requires_grad_(True)
    y = torch.randint(0, V, (T,), generator=g, device=dev)
    up = torch.randn(T, generator=g, device=dev) / T
    lp, _ = ops.lmhead_logprob(h, w, None, y, keep_logits="recompute")
    dh, dw = torch.autograd.grad(lp, (h, w), up)
    hd, wd = h.detach().double(), w.detach().double()
    ds = -torch.softmax(hd @ wd.t(), 1)
    ds[torch.arange(T, device=dev), y] += 1
    ds *= up[:, None].double()
    for got, want in ((dh, ds @ wd), (dw, ds.t() @ hd)):
        assert (got.double() - want).norm() <= 6e-3 * want.norm() + 1e-12
