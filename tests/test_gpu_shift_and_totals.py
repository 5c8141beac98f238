"""GPU tests of the label shift in one launch and of the loss whose block sums the last chunk's preparation adds up."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1,), (7,), (1, 1), (1, 256), (3, 257), (2, 3, 5), (1, 70001), (0, 4)])
def test_label_shift_is_the_padded_slice(dev, shape):
    from fgrpo import ops
    x = torch.randint(-100, 1 << 40, shape, device=dev)
    want = torch.nn.functional.pad(x, (0, 1), value=-100)[..., 1:]
    got = ops.shift_labels(x)
    assert torch.equal(got, want) and got.is_contiguous()
    if x.numel() > 1:
        for view in (x.transpose(0, -1), x[..., ::2], x.int()):          # other layouts and types take the general path
            assert torch.equal(ops.shift_labels(view), torch.nn.functional.pad(view, (0, 1), value=-100)[..., 1:])


@pytest.mark.parametrize("T,chunk", [(1, 256), (300, 256), (4096, 8192), (4097, 1024), (16385, 8192)])
def test_loss_is_the_same_with_and_without_gradients(dev, T, chunk):
    """The launch that closes a step without gradients adds the same block sums in the same order; the token count also
    covers every tile of the pre-pass's sample.  The vocabulary's split may differ between the two: 1e-6."""
    from fgrpo import ops
    g = torch.Generator(device=dev).manual_seed(T)
    h = torch.randn(T, 256, generator=g, device=dev).bfloat16()
    w = (torch.randn(33001, 256, generator=g, device=dev) * 0.05).bfloat16()
    y = torch.randint(0, 33001, (T,), generator=g, device=dev)
    adv, old = torch.randn(T, generator=g, device=dev), torch.full((T,), -10.0, device=dev)
    assert ops.chunked_supported(T, 256, 33001, torch.bfloat16, chunk)
    with torch.no_grad():
        want = ops.fused_grpo_loss(h, w, None, y, old, adv, chunk_tokens=chunk)[0]
    h.requires_grad_(True)
    loss, _, _, _, l1, l2, lp = ops.fused_grpo_loss(h, w, None, y, old, adv, chunk_tokens=chunk)
    x = h.detach().double() @ w.double().t()
    ref = x.gather(1, y[:, None])[:, 0] - torch.logsumexp(x, 1)
    assert (lp - ref).abs().max() <= 4e-5
    assert abs(float(loss.detach()) - float(want)) <= 1e-6 + 1e-6 * abs(float(want))
    dh, = torch.autograd.grad(loss, h)
    assert torch.isfinite(dh).all()
