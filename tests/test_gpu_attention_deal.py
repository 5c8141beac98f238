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
