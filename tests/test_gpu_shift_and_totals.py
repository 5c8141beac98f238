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


def test_label_shift_under_a_function_transform_and_a_trace(dev):
    """Wrapped tensors have the plain type in Python: they, and what a dispatch mode records, take torch's operations."""
    from fgrpo import ops
    from torch.fx.experimental.proxy_tensor import make_fx
    x, y = (torch.randint(-100, 1 << 40, (4, 9), device=dev) for _ in range(2))
    want = lambda t: torch.nn.functional.pad(t, (0, 1), value=-100)[..., 1:]
    assert torch.equal(torch.func.vmap(ops.shift_labels)(x), want(x))
    assert torch.equal(make_fx(ops.shift_labels)(x)(y), want(y))
    assert torch.equal(torch.compile(ops.shift_labels, backend="eager", fullgraph=True)(y), want(y))


def test_label_shift_under_a_function_mode(dev):
    """A trace before dispatch is a function mode and no dispatch mode: it, and any other such mode, sees the operations."""
    from fgrpo import ops
    from torch.fx.experimental.proxy_tensor import make_fx
    from torch.overrides import TorchFunctionMode
    x, y = (torch.randint(-100, 1 << 40, (4, 9), device=dev) for _ in range(2))
    want = lambda t: torch.nn.functional.pad(t, (0, 1), value=-100)[..., 1:]
    assert torch.equal(make_fx(ops.shift_labels, pre_dispatch=True)(x)(y), want(y))
    seen = []

    class Record(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    with Record():
        assert torch.equal(ops.shift_labels(x), want(x))
    assert torch.nn.functional.pad in seen


def test_log_probabilities_without_the_extension_module(dev, monkeypatch):
    """The log-probability entry point needs the library alone; without the module the shift is torch's."""
    import grpo_loss as G
    from fgrpo import _lib, ops
    g = torch.Generator(device=dev).manual_seed(5)
    h, w = torch.randn(1, 70, 64, generator=g, device=dev), torch.randn(999, 64, generator=g, device=dev)
    y = torch.randint(0, 999, (1, 70), generator=g, device=dev)
    with torch.no_grad():
        want = G.fused_log_probs_and_entropy_fn(w, None, h, y)
        monkeypatch.setattr(_lib, "_native", None)
        monkeypatch.setattr(_lib, "BINDING_PATH", _lib.BINDING_PATH + ".absent")
        got = G.fused_log_probs_and_entropy_fn(w, None, h, y)
    assert torch.equal(ops.shift_labels(y), torch.nn.functional.pad(y, (0, 1), value=-100)[..., 1:])
    assert all(torch.equal(a, b) for a, b in zip(got, want))


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


@pytest.mark.parametrize("T,bounds", [(1, [0, 1]), (63, [0, 10, 10, 63]), (1024, [0, 1000, 1024]), (1025, [3, 700, 1020]), (2047, [0, 2047]),
                                      (2048, list(range(0, 2049, 8))), (1500, list(range(0, 641, 10))), (1500, list(range(0, 651, 10))),
                                      (2048, list(range(2049))), (2049, [0, 5, 2049]), (2048, [0, 3000]), (700, [600, 50, 650])])
@pytest.mark.parametrize("mode", ["token_mean", "sample_mean"])
@pytest.mark.parametrize("denom", [0.0, 7.0])
def test_objective_of_a_small_batch(dev, T, bounds, mode, denom):
    """One work-group up to 2048 tokens in 64 segments, three launches beyond: the same formula in fp64 from the same log-probabilities.
    Weights, ratios and products are fp32: a dozen roundings, 2e-6 of the largest term."""
    from fgrpo import ops
    g = torch.Generator(device=dev).manual_seed(T)
    r = lambda s=1.0: torch.randn(T, generator=g, device=dev) * s
    lp, adv = r(0.3) - 3, r()
    old, ref = lp + r(0.2), lp + r(0.2)
    y = torch.randint(0, 9, (T,), generator=g, device=dev)
    y[torch.rand(T, generator=g, device=dev) < 0.3] = -100
    cu = torch.tensor(bounds, dtype=torch.int32, device=dev)
    loss, gr, lr, c1, l1, l2, scal = ops.grpo_loss_fwd(lp, old, ref, adv, y, cu, 0.2, 0.28, 3.0, 0.01, mode, denom)
    on = (y != -100).double()
    w, full = torch.zeros_like(on), 0
    if mode == "sample_mean":
        for a, b in zip(bounds, bounds[1:]):
            a, b = max(a, 0), min(b, T)
            n = float(on[a:b].sum()) if b > a else 0.0
            if n > 0:
                w[a:b], full = 1.0 / n, full + 1
    else:
        w, full = w + 1, float(on.sum())
    den = max(denom if denom > 0 else float(full), 1.0)
    x = lp.double().requires_grad_(True)
    ratio, a = torch.exp(x - old.double()), adv.double()
    u, v = -a * ratio, -a * ratio.clamp(0.8, 1.28)
    m = torch.maximum(u, v)
    tok = torch.where(a < 0, torch.minimum(m, -a * 3.0), m)
    d = ref.double() - x
    tok = tok + 0.01 * (torch.exp(d) - d - 1)
    want = (w * on * tok).sum() / den
    gw, = torch.autograd.grad(want, x)
    big = float((w * on * tok.detach().abs()).sum()) / den + 1e-12
    assert abs(float(loss) - float(want.detach())) <= 2e-6 * big + 1e-9
    assert (gr.double() - gw).abs().max() <= 2e-6 * float(gw.abs().max()) + 1e-12
    assert float(scal[1]) == float(on.sum())


def test_many_segments_are_not_walked_by_one_work_group(dev):
    """A segment costs a wavefront half a microsecond: 2048 of them took one work-group nine times as long as 64; over the
    device they take less than twice as long."""
    from fgrpo import ops
    T = 2048
    lp, adv, y = torch.randn(T, device=dev), torch.randn(T, device=dev), torch.zeros(T, dtype=torch.long, device=dev)

    def us(segments):
        cu = torch.linspace(0, T, segments + 1, device=dev).int()
        call = lambda: ops.grpo_loss_fwd(lp, lp, None, adv, y, cu, 0.2, 0.28, 3.0, 0.0, "sample_mean", 0.0)
        call()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for _ in range(20):
                call()
        best = float("inf")
        for _ in range(5):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            graph.replay()
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b))
        return best
    assert us(T) < 4 * us(64)
