"""GPU tests of token counts just past a whole tile, whose last tokens may take a narrow tile in the forward: contractions
shorter than the loads run ahead, both kinds of input, with and without kept numerators; and, where the plan is asserted to
hold such a tile, both widths' edges with and without whole tiles before it, in the first and the second token region."""
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


# one token region (its last tile alone or behind whole ones), then the second of two: 16384 tokens lie in the first
NARROW = [(1, 33001), (64, 33001), (65, 33001), (128, 33001), (257, 33001), (320, 33001), (833, 33001), (896, 33001),
          (321, 151936), (384, 151936), (868, 151936), (16385, 33001), (16448, 33001), (16449, 33001), (16512, 33001),
          (17153, 33001), (17216, 33001), (17217, 33001), (17280, 33001)]


def takes_a_narrow_tile(T, H, V):
    """Its partials are workspace that the plan without narrow tiles does not have."""
    from fgrpo import _lib
    need = []
    for on in (0, 1):
        _lib.set_tuning(fwd_tail=on)
        need.append(_lib.load().fgrpo_logprob_fwd_workspace(T, H, V, _lib.BF16))
    return need[0] != need[1]


@pytest.mark.parametrize("T,V", NARROW)
def test_narrow_tiles_of_the_forward(dev, T, V):
    """As test_last_tokens_of_the_forward, in rows."""
    from fgrpo import ops
    h, w, y, _ = problem(dev, T, 64, V, torch.bfloat16)
    assert takes_a_narrow_tile(T, 64, V)
    got = ops.lmhead_logprob_fwd(h, w, None, y)
    wd = w.double().t()
    for a in range(0, T, 1024):
        yc = y[a:a + 1024]
        x = h[a:a + 1024].double() @ wd
        lse, on = torch.logsumexp(x, 1), yc >= 0
        lp, ent, got_lse = (t[a:a + 1024] for t in got)
        zero = torch.zeros_like(lse)
        assert (got_lse - lse).abs().max() <= 2e-5
        assert (lp - torch.where(on, x.gather(1, yc.clamp(min=0)[:, None])[:, 0] - lse, zero)).abs().max() <= 4e-5
        x = torch.exp(x - lse[:, None]) * x
        assert (ent - torch.where(on, lse - x.sum(1), zero)).abs().max() <= 4e-5


@pytest.mark.parametrize("T,V", [t for t in NARROW if t[0] in (320, 833, 896, 868, 16385, 16449, 17216, 17280)])
def test_gradients_behind_narrow_tiles(dev, T, V):
    """As test_gradients_of_the_last_tokens, the rows of the last tile on their own too."""
    from fgrpo import ops
    h, w, y, _ = problem(dev, T, 256, V, torch.bfloat16)
    assert takes_a_narrow_tile(T, 256, V) and ops.keep_supported(T, 256, V, torch.bfloat16)
    h.requires_grad_(True), w.requires_grad_(True)
    up = torch.randn(T, device=dev) / T
    lp, _ = ops.lmhead_logprob(h, w, None, y, keep_logits="whole")
    dh, dw = torch.autograd.grad(lp, (h, w), up)
    hd, wd = h.detach().double(), w.detach().double()
    g = torch.where(y >= 0, up, torch.zeros_like(up)).double()
    want_h, want_w = torch.empty_like(hd), torch.zeros_like(wd)
    for a in range(0, T, 1024):
        hc, yc = hd[a:a + 1024], y[a:a + 1024]
        ds = -torch.softmax(hc @ wd.t(), 1)
        ds[torch.arange(len(yc), device=dev), yc.clamp(min=0)] += 1
        ds *= g[a:a + 1024, None]
        want_h[a:a + 1024] = ds @ wd
        want_w += ds.t() @ hc
    last = (T - 1) // 256 * 256
    for got, want in ((dh, want_h), (dh[last:], want_h[last:]), (dw, want_w)):
        assert (got.double() - want).norm() <= 6e-3 * want.norm() + 1e-12
