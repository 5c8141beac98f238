"""GPU tests of attention launches whose tiles are dealt to several work-groups (batches with too few tiles for the
device): against the undivided launches, against the oracle, and twice for reproducibility."""
import pytest
import torch

from oracle import attn_oracle as AO

pytestmark = pytest.mark.gpu

SHAPES = [  # tokens, segment bounds, query heads, K/V heads, head dimension
    (777, [0, 777], 12, 2, 128), (513, [0, 513], 4, 1, 128), (1500, [0, 1500], 14, 2, 64), (1025, [0, 1025], 8, 8, 64),
    (2047, [0, 1024, 1030, 2047], 28, 4, 128), (1990, [0, 3, 900, 1990], 3, 1, 64), (4200, [0, 4200], 2, 1, 128),
    (1300, [0, 1216, 1300], 16, 4, 128), (6000, [0, 6000], 12, 2, 128), (640, [0, 640], 1, 1, 128)]


def operands(T, Hq, Hkv, D, dev):
    g = torch.Generator().manual_seed(T)
    return [torch.randn(T, n, D, generator=g).bfloat16().to(dev) for n in (Hq, Hkv, Hkv, Hq)]


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("T,cu,Hq,Hkv,D", SHAPES)
def test_divided_tiles_agree_with_whole_ones(dev, T, cu, Hq, Hkv, D, causal):
    """Two roundings to bf16 (probabilities, result) of 2^-9 at most on either side: 2^-7 of the norm between them."""
    from fgrpo import _lib, ops
    lib = _lib.load()
    if causal:       # without the mask some of the shapes fill the device as they are
        assert lib.fgrpo_varlen_attn_workspace(T, len(cu) - 1, Hq, Hkv, D, causal, 1) > 0, "this shape is meant to be divided"
    q, k, v, do = operands(T, Hq, Hkv, D, dev)
    cu_t = torch.tensor(cu, dtype=torch.int32, device=dev)
    out0, lse = ops.varlen_attn_fwd(q, k, v, cu_t, None, causal)
    want = (out0,) + tuple(ops.varlen_attn_bwd(do, q, k, v, out0, lse, cu_t, None, causal))

    def once():
        a = [x.clone().requires_grad_(True) for x in (q, k, v)]
        out = ops.varlen_attention(*a, cu_t, None, causal)
        return (out.detach(),) + torch.autograd.grad(out, a, do)
    got, again = once(), once()
    for name, x, y, z in zip(("out", "dq", "dk", "dv"), got, want, again):
        assert torch.equal(x, z), f"{name} is not reproducible"
        assert torch.isfinite(x).all()
        assert (x.float() - y.float()).norm() <= 2 ** -7 * y.float().norm(), name


def test_divided_forward_against_the_oracle(dev):
    from fgrpo import ops
    T, cu, Hq, Hkv, D = SHAPES[4]
    q, k, v, do = operands(T, Hq, Hkv, D, dev)
    cu_t = torch.tensor(cu, dtype=torch.int32, device=dev)
    with torch.no_grad():
        out = ops.varlen_attention(q, k, v, cu_t)
    want = AO.varlen_attention(q.float().cpu(), k.float().cpu(), v.float().cpu(), torch.tensor(cu), causal=True)
    want = want[0] if isinstance(want, tuple) else want
    assert (out.float().cpu() - want).norm() <= 2 ** -8 * want.norm()


def test_workspace_is_checked(dev):
    from fgrpo import _lib
    lib = _lib.load()
    T, Hq, Hkv, D = 777, 12, 2, 128
    q, k, v, _ = operands(T, Hq, Hkv, D, dev)
    cu = torch.tensor([0, T], dtype=torch.int32, device=dev)
    out, lse = torch.empty_like(q), torch.empty(Hq, T, device=dev)
    bounds = torch.empty(4 * T, dtype=torch.int32, device=dev)
    need = lib.fgrpo_varlen_attn_workspace(T, 1, Hq, Hkv, D, 1, 0)
    ws = torch.empty(need, dtype=torch.uint8, device=dev)
    args = [t.data_ptr() for t in (q, k, v)] + [Hq * D, D, Hkv * D, D, Hkv * D, D, cu.data_ptr(), 1, T, Hq, Hkv, D, 0.088, 1,
                                                out.data_ptr(), lse.data_ptr(), bounds.data_ptr(), 0]
    st = torch.cuda.current_stream().cuda_stream
    assert need > 0 and lib.fgrpo_varlen_attn_fwd_ws(*args, ws.data_ptr(), need - 1, st) != 0
    assert lib.fgrpo_varlen_attn_fwd_ws(*args, ws.data_ptr(), need, st) == 0
    assert lib.fgrpo_varlen_attn_fwd_ws(*args, None, 0, st) == 0
    torch.cuda.synchronize()
