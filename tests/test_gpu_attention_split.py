"""GPU tests of attention launches whose tiles are dealt to several work-groups (batches with too few tiles for the
device): against the undivided launches, against the oracle, and twice for reproducibility."""
import pytest
import torch

from oracle import attn_oracle as AO

pytestmark = pytest.mark.gpu

# tokens, segment bounds, query heads, K/V heads, head dimension, and which launches have tiles dealt out (f: forward,
# q: dQ, k: dK/dV) with the causal mask and without
SHAPES = [
    (777, [0, 777], 12, 2, 128, "fqk", "k"), (513, [0, 513], 4, 1, 128, "fqk", "fqk"), (1500, [0, 1500], 14, 2, 64, "fqk", "k"),
    (1025, [0, 1025], 8, 8, 64, "fq", "fq"), (2047, [0, 1024, 1030, 2047], 28, 4, 128, "k", "k"),
    (1990, [0, 3, 900, 1990], 3, 1, 64, "fqk", "q"), (4200, [0, 4200], 2, 1, 128, "fqk", "fqk"),
    (1300, [0, 1216, 1300], 16, 4, 128, "k", ""), (6000, [0, 6000], 12, 2, 128, "fqk", "k"), (640, [0, 640], 1, 1, 128, "fq", "fq")]
CASES = [(*shape[:5], causal, sides) for shape in SHAPES for causal, sides in ((True, shape[5]), (False, shape[6])) if sides]


def divided(T, n_seq, Hq, Hkv, D, causal):
    """Which launches of a call deal tiles out: those that ask for scratch, the backward's two with the other switched to
    a kernel that cannot."""
    from fgrpo import _lib
    need = lambda backward: _lib.load().fgrpo_varlen_attn_workspace(T, n_seq, Hq, Hkv, D, causal, backward) > 0
    found = "f" if need(0) else ""
    try:
        _lib.set_tuning(attn_dkv=1)
        found += "q" if need(1) else ""
        _lib.set_tuning(attn_dkv=0, attn_qside=3)
        found += "k" if need(1) else ""
    finally:
        _lib.set_tuning(attn_dkv=0, attn_qside=0)
    return found


def operands(T, Hq, Hkv, D, dev):
    g = torch.Generator().manual_seed(T)
    return [torch.randn(T, n, D, generator=g).bfloat16().to(dev) for n in (Hq, Hkv, Hkv, Hq)]


@pytest.mark.parametrize("T,cu,Hq,Hkv,D,causal,sides", CASES)
def test_divided_tiles_agree_with_whole_ones(dev, T, cu, Hq, Hkv, D, causal, sides):
    """Two roundings to bf16 (probabilities, result) of 2^-9 at most on either side: 2^-7 of the norm between them."""
    from fgrpo import ops
    assert divided(T, len(cu) - 1, Hq, Hkv, D, causal) == sides
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


@pytest.mark.parametrize("T,cu,Hq,Hkv,D,causal,sides", [c for c in CASES if c[0] < 2000])
def test_divided_tiles_against_the_oracle(dev, T, cu, Hq, Hkv, D, causal, sides):
    """Every launch that is divided (all three at both head dimensions).  Probabilities and results are rounded to bf16,
    2^-9 each: 2^-8 of the norm for the output and dV; dS, from a delta of the rounded output, is rounded once more
    on the way to dQ and dK: 2^-7."""
    from fgrpo import ops
    q, k, v, do = operands(T, Hq, Hkv, D, dev)
    a, o = [[x.clone().to(d, t).requires_grad_(True) for x in (q, k, v)] for d, t in ((dev, torch.bfloat16), ("cpu", torch.float32))]
    got = ops.varlen_attention(*a, torch.tensor(cu, dtype=torch.int32, device=dev), None, causal)
    want = AO.varlen_attention(*o, torch.tensor(cu), causal=causal)
    got, want = (got, *torch.autograd.grad(got, a, do)), (want, *torch.autograd.grad(want, o, do.float().cpu()))
    for name, x, y, tol in zip(("out", "dq", "dk", "dv"), got, want, (2 ** -8, 2 ** -7, 2 ** -7, 2 ** -8)):
        err = ((x.detach().float().cpu() - y.detach()).norm() / y.detach().norm()).item()
        assert err <= tol, name


def lengths(T, lo, hi):
    g = torch.Generator().manual_seed(T + hi)
    out = []
    while sum(out) < T:
        out.append(min(int(torch.randint(lo, hi + 1, (1,), generator=g)), T - sum(out)))
    return out


@pytest.mark.parametrize("T,lens,Hq,Hkv,D", [
    (2000, [2000], 14, 2, 64), (2000, [2000], 12, 2, 128), (2000, lengths(2000, 128, 512), 28, 4, 128),      # all parts in flight at once, none to spare
    (3000, [1916, 200, 700, 184], 12, 2, 128), (3001, lengths(3001, 128, 512), 28, 4, 128),
    (4000, lengths(4000, 128, 1024), 28, 4, 128), (5000, [5000], 28, 4, 128), (9000, lengths(9000, 128, 2048), 12, 2, 128),      # more parts than the device holds
    (9000, lengths(9000, 128, 2048), 14, 2, 64), (9000, [4300, 4700], 8, 2, 128), (1501, [1024, 477], 12, 2, 128), (70, [70], 12, 1, 128), (5, [2, 3], 64, 1, 128)])           # more than 64 tiles an XCD; two tiles; one, left whole
def test_tiles_dealt_by_their_steps_agree_with_whole_ones(dev, T, lens, Hq, Hkv, D):
    """Bounds as in test_divided_tiles_agree_with_whole_ones."""
    from fgrpo import _lib, ops
    q, k, v, do = operands(T, Hq, Hkv, D, dev)
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device=dev)
    out, lse = ops.varlen_attn_fwd(q, k, v, cu, None, True)
    want = ops.varlen_attn_bwd(do, q, k, v, out, lse, cu, None, True)
    assert (_lib.load().fgrpo_varlen_attn_workspace(T, len(lens), Hq, Hkv, D, 1, 1) > 0) == (T > 5)

    def once():
        a = [x.clone().requires_grad_(True) for x in (q, k, v)]
        o = ops.varlen_attention(*a, cu, None, True)
        return (o.detach(),) + torch.autograd.grad(o, a, do)
    for name, x, y, z in zip(("out", "dq", "dk", "dv"), once(), (out, *want), once()):
        assert torch.equal(x, z), f"{name} is not reproducible"
        assert (x.float() - y.float()).norm() <= 2 ** -7 * y.float().norm(), name


@pytest.mark.parametrize("longest", [1694, 1, 10 ** 9, 0, -5, None, 1694.0, torch.tensor(1694)])
def test_the_longest_segment_a_caller_names_decides_no_result(dev, longest):
    """True, wrong, out of range or of another type: bounds as in test_divided_tiles_agree_with_whole_ones."""
    from fgrpo import _lib, ops
    from varlen_attention import flash_attn_varlen_func
    lens, Hq, Hkv, D = [1694, 400] + [300] * 13, 16, 4, 128
    T = sum(lens)
    need = lambda n: _lib.load().fgrpo_varlen_attn_workspace_len(T, len(lens), n, Hq, Hkv, D, 1, 0)
    assert need(1694) > 0 and need(0) == 0 == need(1) and need(10 ** 9) == need(T)
    q, k, v, do = operands(T, Hq, Hkv, D, dev)
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device=dev)
    out, lse = ops.varlen_attn_fwd(q, k, v, cu, None, True)
    want = (out, *ops.varlen_attn_bwd(do, q, k, v, out, lse, cu, None, True))
    a = [x.clone().requires_grad_(True) for x in (q, k, v)]
    o = flash_attn_varlen_func(*a, cu, cu, longest, longest, causal=True)
    for name, x, y in zip(("out", "dq", "dk", "dv"), (o.detach(), *torch.autograd.grad(o, a, do)), want):
        assert (x.float() - y.float()).norm() <= 2 ** -7 * y.float().norm(), name


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
