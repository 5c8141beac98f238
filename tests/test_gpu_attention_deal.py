"""GPU tests of what the attention launches do with tiles dealt to several work-groups beyond agreeing with whole ones."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def operands(T, Hq, Hkv, D, dev):
    g = torch.Generator().manual_seed(T)
    return [torch.randn(T, n, D, generator=g).bfloat16().to(dev) for n in (Hq, Hkv, Hkv, Hq)]


@pytest.mark.parametrize("held", [(8, 2 ** 31 - 1), (8, -1), (8, 4096), (9, 0), (2 ** 31 - 1, 0), (0, 0)])
@pytest.mark.parametrize("T,Hq,Hkv,D", [(70, 12, 1, 128), (128, 12, 1, 128), (777, 12, 2, 128), (513, 4, 1, 64)])
def test_an_order_list_that_leaves_tiles_out_reads_nothing_from_outside_the_workspace(dev, T, Hq, Hkv, D, held):
    """A caller's lists may name one tile again and again.  The other tiles' entries of the merge's table are then whatever
    the workspace held: rows of theirs are not written.  Bounds of the named tile as in test_gpu_attention_split."""
    from fgrpo import _lib, ops
    lib = _lib.load()
    q, k, v, do = operands(T, Hq, Hkv, D, dev)
    cu = torch.tensor([0, T], dtype=torch.int32, device=dev)
    want, lse0 = ops.varlen_attn_fwd(q, k, v, cu, None, True)
    bounds = ops.attention_bounds(cu, T, True)
    bounds[2 * T:] = 0                                        # every list: tile 0, over and over
    p, st = (lambda t: t.data_ptr()), torch.cuda.current_stream().cuda_stream
    shape = [Hq * D, D, Hkv * D, D, Hkv * D, D, p(cu), 1, T, Hq, Hkv, D, D ** -0.5, 1]

    def workspace(backward):
        n = lib.fgrpo_varlen_attn_workspace(T, 1, Hq, Hkv, D, 1, backward)
        return torch.tensor(held, dtype=torch.int32, device=dev).repeat(n // 8).view(torch.uint8) if n else None
    tail = lambda ws: (None, 0, st) if ws is None else (p(ws), ws.numel(), st)
    out, lse = torch.full_like(q, 77.0), torch.full_like(lse0, 77.0)
    assert lib.fgrpo_varlen_attn_fwd_ws(p(q), p(k), p(v), *shape, p(out), p(lse), p(bounds), 1, *tail(workspace(0))) == 0
    torch.cuda.synchronize()
    assert (out[:32].float() - want[:32].float()).norm() <= 2 ** -7 * want[:32].float().norm()      # every tile has 32 tokens or more
    assert (out[128:] == 77.0).all()                                                                  # ... and 128 at most
    dq, dk, dv, delta = torch.full_like(q, 77.0), torch.full_like(k, 77.0), torch.full_like(v, 77.0), torch.zeros_like(lse)
    ws = workspace(1)
    assert ws is not None
    assert lib.fgrpo_varlen_attn_bwd_ws(p(do), p(q), p(k), p(v), p(want), p(lse0), *shape, p(dq), p(dk), p(dv), p(delta), p(bounds), 1, *tail(ws)) == 0
    torch.cuda.synchronize()
    for x in (dq, dk, dv):
        assert (x[128:] == 77.0).all() and (x[:32] != 77.0).any()


def launches(T, n_seq, longest, Hq, Hkv, D, causal):
    """Which launches of a call deal their tiles out, as the call plans them: those that ask for scratch, dQ for what is left of the
    backward's when a kernel that cannot is put in its place."""
    from fgrpo import _lib
    need = lambda backward: _lib.load().fgrpo_varlen_attn_workspace_len(T, n_seq, longest, Hq, Hkv, D, causal, backward)
    found, both = "f" if need(0) else "", need(1)
    try:
        _lib.set_tuning(attn_qside=3)
        keys = need(1)
    finally:
        _lib.set_tuning(attn_qside=0)
    return found + ("q" if both > keys else "") + ("k" if keys else "")


# segment lengths, query heads, K/V heads, head dimension, mask, which launches (f: forward, q: dQ, k: dK/dV) are dealt out; 1, 2 and 4
# heads a work-group and one to five work-groups a group, all parts in flight or more than the device holds
DEALT = [
    ([1216, 84], 16, 4, 128, True, "fqk"), ([1500, 300, 40, 560, 200], 12, 2, 128, True, "fqk"), ([1500, 300, 40, 560, 200], 15, 3, 64, True, "fqk"),
    ([1694] + [400] * 10 + [100, 206], 16, 4, 128, True, "fqk"), ([1500, 300, 40, 560, 200], 28, 4, 128, True, "qk"), ([9000], 5, 1, 128, True, "fqk"),
    ([300, 4000, 1700, 1000, 1900, 100], 6, 3, 128, True, "fqk"), ([8200, 3000, 100, 1700, 3000], 8, 8, 64, True, "fq"),
    ([1, 1700, 1299, 400, 500, 100], 12, 6, 128, True, "fqk"), ([12000, 8000], 3, 1, 128, True, "fqk"),
    ([700], 5, 1, 128, False, "fqk"), ([1216, 84], 3, 1, 128, False, "fqk"), ([9000], 3, 1, 128, False, "fqk"), ([700], 4, 4, 128, False, "fq"),
    ([1500, 300, 700, 1500], 2, 1, 128, False, "fq"), ([10, 2900, 40, 3000, 2050], 1, 1, 64, False, "fq"), ([300, 4000, 1700, 1000, 1900, 100], 5, 1, 128, False, "k"),
    ([1500, 300, 40, 560, 200], 12, 2, 128, False, "k")]


@pytest.mark.parametrize("lens,Hq,Hkv,D,causal,sides", DEALT)
def test_the_launches_meant_are_dealt_out_and_agree_with_whole_ones(dev, lens, Hq, Hkv, D, causal, sides):
    """With the longest segment named.  Two roundings to bf16 (probabilities, result) of 2^-9 at most on either side: 2^-7 of the
    norm between them."""
    from fgrpo import ops
    T = sum(lens)
    assert launches(T, len(lens), max(lens), Hq, Hkv, D, causal) == sides
    q, k, v, do = operands(T, Hq, Hkv, D, dev)
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device=dev)
    out, lse = ops.varlen_attn_fwd(q, k, v, cu, None, causal)
    want = (out, *ops.varlen_attn_bwd(do, q, k, v, out, lse, cu, None, causal))

    def once():
        a = [x.clone().requires_grad_(True) for x in (q, k, v)]
        o = ops.varlen_attention(*a, cu, None, causal, None, max(lens))
        return (o.detach(),) + torch.autograd.grad(o, a, do)
    for name, x, y, z in zip(("out", "dq", "dk", "dv"), once(), want, once()):
        assert torch.equal(x, z), f"{name} is not reproducible"
        assert (x.float() - y.float()).norm() <= 2 ** -7 * y.float().norm(), name


def test_dealt_out_launches_are_capturable(dev):
    """All three launches dealt out, their tables and sums written anew by every replay: same bits as an eager call on the inputs at hand."""
    from fgrpo import ops
    lens, Hq, Hkv, D = [1500, 300, 40, 560, 200], 12, 2, 128
    T = sum(lens)
    assert launches(T, len(lens), max(lens), Hq, Hkv, D, True) == "fqk"
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device=dev)
    q, k, v, do = operands(T, Hq, Hkv, D, dev)
    q, k, v = (x.requires_grad_(True) for x in (q, k, v))

    def once():
        o = ops.varlen_attention(q, k, v, cu, None, True, None, max(lens))
        return (o.detach(),) + torch.autograd.grad(o, (q, k, v), do)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        once()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        held = once()
    for seed in range(3):
        with torch.no_grad():
            for x in (q, k, v, do):
                x.copy_(torch.randn(x.shape, generator=torch.Generator().manual_seed(seed)))
        want = once()
        graph.replay()
        torch.cuda.synchronize()
        for name, x, y in zip(("out", "dq", "dk", "dv"), held, want):
            assert torch.equal(x, y), (seed, name)
