"""GPU tests of what small and prompt-heavy batches take: the merge of finely split vocabularies, evaluation without
a gradient, and the log-probability worker's skipping of masked positions."""
import pytest
import torch

from test_gpu_dropin import TinyLM, make_samples

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,V,H", [(1, 131, 64), (15, 4099, 64), (17, 40000, 128), (300, 40000, 64), (513, 70001, 64)])
def test_vocabulary_splits_are_merged_at_every_count(dev, T, V, H):
    """From one split to many more than a token has threads; against the soft-max in fp32 on the same bf16 operands.
    Tolerance: fp32 sums over V terms in another order, a few ulp of values below 16."""
    from fgrpo import ops
    g = torch.Generator().manual_seed(T)
    h = torch.randn(T, H, generator=g).bfloat16().to(dev)
    w = (torch.randn(V, H, generator=g) * 0.1).bfloat16().to(dev)
    y = torch.randint(0, V, (T,), generator=g).to(dev)
    lp, ent, lse = ops.lmhead_logprob_fwd(h, w, None, y)
    x = h.float() @ w.float().t()
    want = torch.logsumexp(x, 1)
    p = torch.softmax(x, 1)
    assert (lse - want).abs().max() <= 2e-5
    assert (lp - (x.gather(1, y[:, None])[:, 0] - want)).abs().max() <= 4e-5
    assert (ent - (want - (p * x).sum(1))).abs().max() <= 4e-5


def test_evaluation_of_a_trainable_head_prepares_no_backward(dev):
    """Under no_grad the results are those of the differentiable call and carry no graph."""
    from fgrpo import ops
    g = torch.Generator().manual_seed(0)
    h = torch.randn(700, 1024, generator=g).bfloat16().to(dev).requires_grad_(True)
    w = (torch.randn(9000, 1024, generator=g) * 0.02).bfloat16().to(dev).requires_grad_(True)
    y = torch.randint(0, 9000, (700,), generator=g).to(dev)
    old, adv = torch.randn(700, generator=g).to(dev) - 9, torch.randn(700, generator=g).to(dev)
    lp, ent = ops.lmhead_logprob(h, w, None, y)
    step = ops.fused_grpo_loss(h, w, None, y, old, adv)
    with torch.no_grad():
        lp0, ent0 = ops.lmhead_logprob(h, w, None, y)
        step0 = ops.fused_grpo_loss(h, w, None, y, old, adv)
    assert lp.requires_grad and step[0].requires_grad and not lp0.requires_grad and not step0[0].requires_grad
    assert torch.equal(lp.detach(), lp0) and torch.equal(ent, ent0)
    for a, b in zip(step, step0):
        assert torch.allclose(a.detach(), b, rtol=1e-5, atol=1e-6)      # the chunked step may split the vocabulary otherwise


def test_logprob_worker_skips_prompts_and_returns_the_same(dev):
    """A prompt-heavy batch above the size from which masked rows are left out: the same values where a label is
    scored, zeros elsewhere."""
    from fgrpo import ops
    from grpo_loss import make_grpo_forward
    from workers import LogProbHarness
    torch.manual_seed(0)
    model = TinyLM(tied=False).to(dev).bfloat16()
    make_grpo_forward(model, mode="eval")
    harness = LogProbHarness(model, dev)
    samples = make_samples(n=130)
    assert sum(len(s["sample_ids"]) for s in samples) >= ops.COMPACT_MIN_TOKENS
    got = harness.compute_log_probs_from_samples(samples, packed=True).buffer.clone()
    keep, ops.COMPACT_MIN_TOKENS = ops.COMPACT_MIN_TOKENS, 1 << 30
    try:
        want = harness.compute_log_probs_from_samples(samples, packed=True).buffer
    finally:
        ops.COMPACT_MIN_TOKENS = keep
    assert torch.equal(got == 0, want == 0)
    assert (got - want).abs().max() <= 2e-5


def test_forward_mode_tangents_are_refused(dev):
    """No node implements forward-mode derivatives; a call that needs no backward must not drop a tangent in silence."""
    import torch.autograd.forward_ad as fwAD
    from fgrpo import ops
    cu = torch.tensor([0, 40], dtype=torch.int32, device=dev)
    q, k, v = (torch.randn(40, n, 64, device=dev).bfloat16() for n in (4, 2, 2))
    h, w = torch.randn(70, 64, device=dev).bfloat16(), torch.randn(300, 64, device=dev).bfloat16()
    y = torch.randint(0, 300, (70,), device=dev)
    idx = torch.arange(0, 70, 2, device=dev)
    with fwAD.dual_level(), torch.no_grad():
        dq, dh = fwAD.make_dual(q, torch.ones_like(q)), fwAD.make_dual(h, torch.ones_like(h))
        for call in (lambda: ops.varlen_attention(dq, k, v, cu), lambda: ops.lmhead_logprob(dh, w, None, y),
                     lambda: ops.fused_grpo_loss(dh, w, None, y, None, torch.ones(70, device=dev), compact=idx),
                     lambda: ops.fused_grpo_loss(dh, w, None, y, None, torch.ones(70, device=dev))):
            with pytest.raises(RuntimeError, match="(?i)jvp"):
                call()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,V,ld", [(1, 5, 8), (3, 2048, 2048), (5, 8191, 8192), (2, 8200, 8208), (4, 10247, 10247), (3, 16392, 16400)])
def test_row_kernels_at_the_edges_of_their_strides(dev, dtype, N, V, ld):
    """Log-probabilities, entropy and gradient on rows that end inside a chunk, a stride of one or four chunks, or are
    not 16-byte aligned; one row ignored.  Against fp64; fp32 sums over V terms, bf16 results rounded to 2^-8."""
    from fgrpo import ops
    g = torch.Generator().manual_seed(V)
    store = (torch.randn(N, ld, generator=g) * 3).to(dtype)
    x = store.to(dev)[:, :V]
    y = torch.randint(0, V, (N,), generator=g)
    y[0] = V - 1
    if N > 1:
        y[1] = -100
    lp, ent, lse = ops.logits_logprob_entropy(x, y.to(dev), -100)
    gt = torch.randn(N, generator=g)
    dx = ops.logits_logprob_bwd(x, y.to(dev), -100, gt.to(dev), lse).cpu().double()
    xd = store[:, :V].double()
    ls = torch.log_softmax(xd, 1)
    live = (y >= 0).double()
    want_lp = ls.gather(1, y.clamp(min=0)[:, None])[:, 0] * live
    want_dx = (torch.nn.functional.one_hot(y.clamp(min=0), V) - ls.exp()) * (gt.double() * live)[:, None]
    assert (lp.cpu().double() - want_lp).abs().max() <= 1e-5
    assert (ent.cpu().double() + (ls.exp() * ls).sum(1)).abs().max() <= 2e-5
    tol = (2 ** -8 if dtype == torch.bfloat16 else 2e-6) * want_dx.abs() + 1e-6 * gt.double().abs()[:, None]
    assert ((dx - want_dx).abs() <= tol).all()


@pytest.mark.parametrize("a_km", [True, False])
@pytest.mark.parametrize("M,N", [(1, 1), (128, 256), (129, 128), (256, 129), (100, 40), (384, 640), (300, 200)])
def test_gradient_products_on_tiles_with_a_half_outside(dev, M, N, a_km):
    """Rows or columns that fill at most half of the last 256-wide tile: the wavefronts of the other half only load.
    Against fp64 on the same bf16 operands: fp32 sums of K = 448 products of order one."""
    from fgrpo import ops
    K = 448
    g = torch.Generator().manual_seed(M * 1000 + N)
    Mp, Np = (M + 255) // 256 * 256, (N + 255) // 256 * 256
    A = torch.randn(K, Mp, generator=g).bfloat16() if a_km else torch.randn(M, K, generator=g).bfloat16()
    B = torch.randn(N, K, generator=g).bfloat16() if a_km else torch.randn(K, Np, generator=g).bfloat16()
    out = ops.gemm_kmajor(A.to(dev), B.to(dev), a_km, not a_km, M, N, K).cpu().double()
    Ad, Bd = (A[:, :M].double().t(), B.double()) if a_km else (A.double(), B[:, :N].double().t())
    assert (out - Ad @ Bd.t()).abs().max() <= 2e-4


@pytest.mark.parametrize("T,H,V", [(100, 64, 500), (1, 64, 4099), (129, 96, 8000), (643, 64, 1000), (2000, 256, 777), (700, 72, 3001)])
def test_fp32_gradients_of_small_heads(dev, T, H, V):
    """Both gradients with the contraction in pieces, over segments of 64 and ragged ends.  Against fp64; products of
    operands split into two bf16 halves: 2^-16 of the norm each way, tripled for the sums of dLogits' own error."""
    from fgrpo import ops
    g = torch.Generator().manual_seed(T + V)
    h, w = torch.randn(T, H, generator=g), torch.randn(V, H, generator=g) * 0.1
    y = torch.randint(0, V, (T,), generator=g)
    gt = torch.randn(T, generator=g)
    hd, wd = h.double().requires_grad_(True), w.double().requires_grad_(True)
    lp = torch.log_softmax(hd @ wd.t(), 1).gather(1, y[:, None])[:, 0]
    want = torch.autograd.grad(lp, (hd, wd), gt.double())
    hg, wg = h.to(dev).requires_grad_(True), w.to(dev).requires_grad_(True)
    got = torch.autograd.grad(ops.lmhead_logprob(hg, wg, None, y.to(dev))[0], (hg, wg), gt.to(dev))
    for a, b in zip(got, want):
        assert (a.cpu().double() - b).norm() <= 6 * 2 ** -16 * b.norm()


@pytest.mark.parametrize("panel_elems", [0, 643 * 256])
@pytest.mark.parametrize("T,H,V", [(643, 64, 1000), (129, 96, 8000), (2000, 256, 777)])
def test_fp32_gradients_do_not_depend_on_which_are_wanted(dev, T, H, V, panel_elems):
    """The two products share launches where both are contracted in pieces; their sums are the same alone, bit for bit,
    and with the vocabulary in several panels."""
    from fgrpo import ops
    gen = torch.Generator().manual_seed(T + V)
    h, w = torch.randn(T, H, generator=gen).to(dev), (torch.randn(V, H, generator=gen) * 0.05).to(dev)
    y = torch.randint(0, V, (T,), generator=gen).to(dev)
    g = torch.randn(T, generator=gen).to(dev)
    lse = torch.logsumexp(h.double() @ w.double().t(), 1).float()
    dh, dw, _ = ops.lmhead_bwd(h, w, None, y, lse, g, None, 1.0, True, True, False, panel_elems)
    only_h, none, _ = ops.lmhead_bwd(h, w, None, y, lse, g, None, 1.0, True, False, False, panel_elems)
    assert none is None and torch.equal(only_h, dh)
    none, only_w, _ = ops.lmhead_bwd(h, w, None, y, lse, g, None, 1.0, False, True, False, panel_elems)
    assert none is None and torch.equal(only_w, dw)


@pytest.mark.parametrize("T,bounds", [(643, [0, 40, 41, 41, 643]), (9000, [5, 100, 8000]), (4097, [0, 4097]), (4096, [4095, 4096]),
                                      (300, [0, 100, 300, 0]), (300, [200, 50]), (300, [-7, 20, 400]), (1, [0, 0]),
                                      (300, [250, 20, 90, 0]), (5000, [4900, 100, 4400, 3, 90, 0])])
def test_segment_weights_cover_every_token(dev, T, bounds):
    """1 / (scored tokens of the sample), zero outside every sample: boundaries that start late, end early, repeat, leave
    the batch or run backwards."""
    from fgrpo import ops
    gen = torch.Generator().manual_seed(T)
    y = torch.randint(0, 9, (T,), generator=gen)
    y[torch.rand(T, generator=gen) < 0.3] = -100
    want = torch.zeros(T)
    filled = 0
    for b, e in zip(bounds[:-1], bounds[1:]):
        b = min(max(b, 0), T)
        e = min(max(e, b), T)
        n = int((y[b:e] != -100).sum())
        want[b:e] = 1.0 / n if n else 0.0
        filled += n > 0
    junk = torch.full((64, T), float("nan"), device=dev)      # what the next allocations may be cut from
    del junk
    tokw, pre = ops.loss_prepare(y.to(dev), torch.tensor(bounds, dtype=torch.int32), "sample_mean")
    assert torch.equal(tokw.cpu(), want)
    assert pre.tolist()[:3] == [max(filled, 1), int((y != -100).sum()), filled]


@pytest.mark.parametrize("compact", [False, True])
@pytest.mark.parametrize("which", ["old_lp", "adv", "ref_lp"])
def test_per_token_inputs_are_inputs_of_the_node(dev, which, compact):
    """They take no gradient, but autograd sees them: a forward-mode tangent is refused with and without gradients, and
    one that requires a gradient gives a loss that does (and a backward that leaves it none)."""
    import torch.autograd.forward_ad as fwAD
    from fgrpo import ops
    h, w = torch.randn(70, 64, device=dev).bfloat16(), torch.randn(300, 64, device=dev).bfloat16()
    y = torch.randint(0, 300, (70,), device=dev)
    tok = dict(old_lp=torch.randn(70, device=dev) - 6, adv=torch.randn(70, device=dev), ref_lp=torch.randn(70, device=dev) - 6)
    extra = dict(kl_beta=0.01, compact=torch.arange(0, 70, 2, device=dev) if compact else False)

    def call(hidden, **over):
        t = dict(tok, **over)
        return ops.fused_grpo_loss(hidden, w, None, y, t["old_lp"], t["adv"], t["ref_lp"], **extra)
    plain = call(h)
    leaf = tok[which].clone().requires_grad_(True)
    out = call(h, **{which: leaf})
    assert not plain[0].requires_grad and out[0].requires_grad and torch.equal(out[0].detach(), plain[0])
    out[0].backward()
    assert leaf.grad is None
    for hidden in (h, h.clone().requires_grad_(True)):
        with fwAD.dual_level():
            dual = fwAD.make_dual(tok[which], torch.ones_like(tok[which]))
            with pytest.raises(RuntimeError, match="(?i)jvp"):
                call(hidden, **{which: dual})
            with torch.no_grad(), pytest.raises(RuntimeError, match="(?i)jvp"):
                call(hidden, **{which: dual})


@pytest.mark.parametrize("entry", ["varlen_attention", "fused_step"])
def test_native_calls_release_the_interpreter_lock(dev, entry):
    """With a switch interval nobody waits out, another thread runs only while a call of this one has let go of the
    lock: it must get on again and again in a row of native calls."""
    import sys
    import threading
    import time
    from fgrpo import _lib
    native = _lib.native()
    cu = torch.tensor([0, 600], dtype=torch.int32, device=dev)
    q, k, v = (torch.randn(600, n, 128, device=dev).bfloat16() for n in (4, 2, 2))
    h, w = torch.randn(600, 256, device=dev).bfloat16(), torch.randn(3000, 256, device=dev).bfloat16()
    y, tok = torch.randint(0, 3000, (600,), device=dev), torch.randn(600, device=dev)
    if entry == "varlen_attention":
        def call():
            return native.varlen_attention(q, k, v, cu, None, True, None)
    else:
        def call():
            return native.fused_step(h, w, None, y, tok, tok, None, None, 1.0, 0.2, 0.2, 3.0, 0.0, False, 0.0, 0, 0, 256, 0)
    with torch.no_grad():
        call()
        torch.cuda.synchronize()
        ran, stop = [0], threading.Event()

        def other():
            while not stop.is_set():
                ran[0] += 1
                time.sleep(2e-4)              # gives the lock up by itself

        interval = sys.getswitchinterval()
        thread = threading.Thread(target=other)
        thread.start()
        sys.setswitchinterval(1000.0)
        try:
            time.sleep(0.05)                  # from here on its waits for the lock are of the long kind
            before, got_on, calls, kept = ran[0], 0, 0, []       # kept: a tensor's end may release the lock too
            while calls < 4000 and got_on < 20:
                kept.append(call())
                got_on += ran[0] > before
                before = ran[0]
                calls += 1
        finally:
            sys.setswitchinterval(interval)
            stop.set()
            thread.join()
            torch.cuda.synchronize()
    # most calls are too short for the other thread to wake in
    print(f"[lock] {entry}: the other thread got on during {got_on} of {calls} calls", flush=True)
    assert got_on == 20


@pytest.mark.parametrize("wrapped", [False, True])
def test_logprob_worker_runs_any_model_of_the_four_inputs(dev, wrapped):
    """The list of scored rows goes to forwards that take it, through a wrapper too; a model with a forward of its own
    gets the four inputs and nothing else, however prompt-heavy the batch."""
    from types import SimpleNamespace
    from fgrpo import ops
    from grpo_loss import make_grpo_forward
    from workers import LogProbHarness

    class Wrapper(torch.nn.Module):
        def __init__(self, inner):
            super().__init__()
            self.module = inner

        def forward(self, *args, **kwargs):
            got.update(kwargs)
            return self.module(*args, **kwargs)

    class Narrow(Wrapper):
        def forward(self, input_ids, attention_mask, position_ids, labels):
            return self.module(input_ids=input_ids, attention_mask=attention_mask, position_ids=position_ids, labels=labels)

    class Own(torch.nn.Module):
        def forward(self, input_ids, attention_mask, position_ids, labels):
            return SimpleNamespace(loss=input_ids.float().view(-1), entropy=position_ids.float().view(-1))
    got = {}
    samples = make_samples(n=130)
    assert sum(len(s["sample_ids"]) for s in samples) >= ops.COMPACT_MIN_TOKENS
    own = Wrapper(Own()) if wrapped else Own()
    res = LogProbHarness(own, dev).compute_log_probs_from_samples(samples)
    assert [r["logprobs"] for r in res] == [[float(t) for t in s["sample_ids"]] for s in samples]
    torch.manual_seed(0)
    model = make_grpo_forward(TinyLM(tied=False).to(dev).bfloat16(), mode="eval")
    LogProbHarness(Wrapper(model), dev).compute_log_probs_from_samples(samples)
    assert "compact_masked_tokens" in got
    LogProbHarness(Narrow(model), dev).compute_log_probs_from_samples(samples)


@pytest.mark.parametrize("trainable", [False, True])
@pytest.mark.parametrize("compact", [False, True])
def test_fused_step_returns_a_tuple_on_every_path(dev, compact, trainable):
    """As every autograd node written in Python does: callers test for it, add to it, use it as a key."""
    from fgrpo import ops
    h, w = (torch.randn(n, 64, device=dev).bfloat16().requires_grad_(trainable) for n in (70, 300))
    out = ops.fused_grpo_loss(h, w, None, torch.randint(0, 300, (70,), device=dev), torch.randn(70, device=dev),
                              torch.randn(70, device=dev), compact=torch.arange(0, 70, 2, device=dev) if compact else False)
    assert type(out) is tuple and len(out) == 7


@pytest.mark.parametrize("trainable", [False, True])
@pytest.mark.parametrize("call", ["fused", "fused_rows", "logprob", "attention"])
def test_traced_calls_run_the_kernels(dev, call, trainable):
    """A trace replays the call on new inputs, with its gradients: results of the eager call, bit for bit (the batch is
    too small for divided tiles)."""
    from fgrpo import ops
    g = torch.Generator().manual_seed(5)
    rand = lambda *shape: torch.randn(*shape, generator=g).to(dev)
    y = torch.randint(0, 300, (70,), generator=g).to(dev)
    tok, cu, rows = (rand(70) - 6, rand(70)), torch.tensor([0, 30, 70], dtype=torch.int32, device=dev), torch.arange(0, 70, 2, device=dev)
    f = dict(fused=lambda a, b: ops.fused_grpo_loss(a, b, None, y, *tok),
             fused_rows=lambda a, b: ops.fused_grpo_loss(a, b, None, y, *tok, compact=rows),
             logprob=lambda a, b: ops.lmhead_logprob(a, b, None, y),
             attention=lambda a, b: ops.varlen_attention(a, b, b, cu))[call]
    shapes = ((70, 4, 64), (70, 2, 64)) if call == "attention" else ((70, 64), (300, 64))

    def leaves():
        return [rand(*s).bfloat16().requires_grad_(trainable) for s in shapes]
    traced = torch.jit.trace(f, tuple(leaves()), check_trace=False)
    args = leaves()
    whole = lambda out: out if isinstance(out, tuple) else (out,)
    want, got = whole(f(*args)), whole(traced(*args))
    assert len(want) == len(got) and all(torch.equal(a, b) for a, b in zip(got, want))
    assert got[0].requires_grad == trainable
    if trainable:
        up = rand(want[0].numel()).to(want[0].dtype).view_as(want[0])
        for a, b in zip(torch.autograd.grad(got[0], args, up), torch.autograd.grad(want[0], args, up)):
            assert torch.equal(a, b)


def test_host_operands_are_refused(dev):
    """Operands beside the ones that decide the device: an address in host memory, or labels for fewer rows than there
    are, must end in an error before anything is launched."""
    from fgrpo import ops
    y, lp, old, adv = torch.randint(0, 300, (70,), device=dev), *(torch.randn(70, device=dev) for _ in range(3))
    h, w = torch.randn(70, 64, device=dev).bfloat16(), torch.randn(300, 64, device=dev).bfloat16()
    rows, logits = torch.arange(0, 70, 2, device=dev), torch.randn(70, 300, device=dev)
    for call in (lambda: ops.grpo_loss_from_logprobs(lp, y, old.cpu(), adv),
                 lambda: ops.grpo_loss_from_logprobs(lp, y, old, adv, ref_lp=old.cpu(), kl_beta=0.1),
                 lambda: ops.fused_grpo_loss(h, w, None, y, old.cpu(), adv),
                 lambda: ops.fused_grpo_loss(h, w, None, y, old.cpu(), adv, compact=rows),
                 lambda: ops.logits_logprob_entropy(logits, y.cpu(), None),
                 lambda: ops.logits_logprob_bwd(logits, y, None, lp.cpu(), lp),
                 lambda: ops.grpo_metrics(rows, lp, old.cpu(), None, adv, lp, lp, 0.2, 0.2)):
        with pytest.raises(RuntimeError, match="must live on the GPU"):
            call()


def test_labels_for_fewer_rows_than_there_are_are_refused(dev):
    from fgrpo import ops
    y, lp, logits = torch.randint(0, 300, (70,), device=dev), torch.randn(70, device=dev), torch.randn(70, 300, device=dev)
    with pytest.raises(RuntimeError, match="69 labels for 70 rows"):
        ops.logits_logprob_entropy(logits, y[:69], None)
    with pytest.raises(RuntimeError, match="69 labels for 70 rows"):
        ops.logits_logprob_bwd(logits, y[:69], None, lp, lp)


@pytest.mark.parametrize("wrong,message", [
    (lambda o: dict(labels=o["labels"][:69]), "one entry per token"),
    (lambda o: dict(old_lp=o["old_lp"][:69]), "old_logprobs has 69 elements"),
    (lambda o: dict(adv=o["adv"][:69]), "advantages has 69 elements"),
    (lambda o: dict(ref_lp=o["adv"][:69]), "ref_logprobs has 69 elements"),
    (lambda o: dict(bias=o["weight"][:299, 0]), "bias must have V elements"),
    (lambda o: dict(weight=o["weight"][:, :63]), "mismatch"),
    (lambda o: dict(weight=o["weight"].float()), "share a dtype"),
    (lambda o: dict(hidden=o["hidden"].half(), weight=o["weight"].half()), "bf16 and fp32 only"),
    (lambda o: dict(adv=o["adv"].cpu()), "must live on the GPU"),
    (lambda o: dict(labels=o["labels"].cpu()), "must live on the GPU"),
    (lambda o: dict(loss_agg_mode="sample_mean"), "needs cu_seqlens"),
    (lambda o: dict(keep_logits="chunked"), "is not supported")])
def test_native_step_refuses_operands_that_do_not_fit(dev, wrong, message):
    """The node in C++ takes its operands' addresses itself: each of its checks must end the call before a launch."""
    from fgrpo import ops
    at = dict(hidden=torch.randn(70, 64, device=dev).bfloat16(), weight=torch.randn(300, 64, device=dev).bfloat16(), bias=None,
              labels=torch.randint(0, 300, (70,), device=dev), old_lp=torch.randn(70, device=dev), adv=torch.randn(70, device=dev))
    at.update(wrong(at))
    operands = [at.pop(name) for name in ("hidden", "weight", "bias", "labels", "old_lp", "adv")]
    operands[0].requires_grad_(True)
    with pytest.raises(RuntimeError, match=message):
        ops.fused_grpo_loss(*operands, **at)
