"""GPU tests of token counts just past a whole tile, whose last tokens take a narrow tile in the forward: every width's
edges, contractions shorter than the loads run ahead, both kinds of input, with and without kept numerators."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def problem(dev, T, H, V, dtype):
    g = torch.Generator(device=dev).manual_seed(T * 7 + H)
    h = torch.randn(T, H, generator=g, device=dev).to(dtype)
    w = (torch.randn(V, H, generator=g, device=dev) * (2.0 / H) ** 0.5).to(dtype)
    y = torch.randint(0, V, (T,), generator=g, device=dev)
    y[torch.arange(0, T, 7, device=dev)] = -100
    return h, w, y, torch.randn(V, generator=g, device=dev).to(dtype) * 0.3


@pytest.mark.parametrize("T", [1, 16, 64, 65, 128, 129, 257, 320, 321, 384, 385, 1033])
@pytest.mark.parametrize("H,dtype,bias", [(64, torch.bfloat16, False), (192, torch.bfloat16, True), (128, torch.float32, False)])
def test_last_tokens_of_the_forward(dev, T, H, dtype, bias):
    """Against the soft-max in fp64 of the same operands; logits stay below 16, so fp32 sums differ by a few ulp of
    that, and split bf16 halves of fp32 inputs by 2^-16 of each product."""
    from fgrpo import ops
    h, w, y, b = problem(dev, T, H, 33001, dtype)
    lp, ent, lse = ops.lmhead_logprob_fwd(h, w, b if bias else None, y)
    x = h.double() @ w.double().t() + (b.double() if bias else 0)
    want, on = torch.logsumexp(x, 1), y >= 0
    p = torch.softmax(x, 1)
    tol = 2e-5 if dtype == torch.bfloat16 else 4e-5
    assert (lse - want).abs().max() <= tol
    zero = torch.zeros_like(want)
    assert (lp - torch.where(on, x.gather(1, y.clamp(min=0)[:, None])[:, 0] - want, zero)).abs().max() <= 2 * tol
    assert (ent - torch.where(on, want - (p * x).sum(1), zero)).abs().max() <= 2 * tol


@pytest.mark.parametrize("T", [16, 65, 129, 300, 321, 385, 777])
def test_gradients_of_the_last_tokens(dev, T):
    """From the numerators a narrow tile keeps, against fp64.  A kept numerator, the scaled hidden row (dW) or the weight
    (dH) and the stored gradient are bf16: 2^-9 each of the norm at most, 6e-3 together."""
    from fgrpo import ops
    h, w, y, _ = problem(dev, T, 256, 33001, torch.bfloat16)
    assert ops.keep_supported(T, 256, 33001, torch.bfloat16)
    h.requires_grad_(True), w.requires_grad_(True)
    up = torch.randn(T, device=dev) / T
    lp, _ = ops.lmhead_logprob(h, w, None, y, keep_logits="whole")
    dh, dw = torch.autograd.grad(lp, (h, w), up)
    g = torch.where(y >= 0, up, torch.zeros_like(up)).double()
    hd, wd = h.detach().double(), w.detach().double()
    ds = -torch.softmax(hd @ wd.t(), 1)
    ds[torch.arange(T, device=dev), y.clamp(min=0)] += 1
    ds *= g[:, None]
    for got, want in ((dh, ds @ wd), (dw, ds.t() @ hd)):
        assert (got.double() - want).norm() <= 6e-3 * want.norm() + 1e-12
