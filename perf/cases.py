"""The workloads this package is timed on: each case is one pass through a public entry point, the way a trainer,
a log-probability worker or a model layer calls it, on inputs of the shapes and distributions such a program has.

Shapes are the package's own benchmark configurations (hidden 896 / 1536 / 3584 / 5120 / 8192, vocabularies of about
128k and 152k, packed samples of 128..1024 or up to 8192 tokens) over the token counts a packed micro-batch really
has: one sample, a partly filled budget, the 36000-token default budget, the benchmark's 32768."""
import math
import os
import random
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "async-grpo-nccl_amd")     # the directory name is not an importable package name
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import grpo_loss as G                                        # noqa: E402
import workers as W                                          # noqa: E402
from varlen_attention import flash_attn_varlen_func          # noqa: E402

IGNORE = -100
GROUP = 8                       # samples of one prompt, whose rewards are normalised together


# ------------------------------------------------------------------------------------------------ the list
def listed():
    return [
        # fp32 training step of the smallest configuration: 16 short samples, tiny head; launches and host work
        _step("step_fp32_anchor", dtype="fp32", tokens=643, H=64, V=1000, lo=16, hi=64, kl=0.001, agg="sample_mean", chunk=0),
        # a micro-batch that holds a single sample of a 1.5B-class policy (tail of a mini-batch, long-tailed packing)
        _step("step_one_sample", dtype="bf16", tokens=777, H=1536, V=151936, lo=777, hi=777, kl=0.0, agg="token_mean", chunk=4096),
        # the benchmark's training step: 1.5B-class policy, 32768 packed tokens, KL to a reference policy
        _step("step_packed_1p5b", dtype="bf16", tokens=32768, H=1536, V=151936, lo=128, hi=1024, kl=0.001, agg="sample_mean", chunk=4096),
        # a full token budget of a 7B-class policy, off every tile boundary, in the plain token-mean objective
        _step("step_budget_7b", dtype="bf16", tokens=35871, H=3584, V=152064, lo=256, hi=8192, kl=0.0, agg="token_mean", chunk=8192),
        # reference-policy log-probabilities of a 32B-class head: forward only, no gradient
        _logprob("logprob_32b", tokens=40000, H=5120, V=152064, lo=1024, hi=4096),
        # one attention layer in training, 1.5B-class heads, the benchmark's packing of short samples
        _attn("attn_packed_12h", tokens=32768, lo=128, hi=1024, Hq=12, Hkv=2, D=128, train=True),
        # one attention layer in training on long samples, 7B-class heads
        _attn("attn_long_28h", tokens=32768, lo=8192, hi=8192, Hq=28, Hkv=4, D=128, train=True),
        # head dimension 64 (0.5B-class heads), a partly filled budget of ragged samples
        _attn("attn_packed_d64", tokens=12345, lo=128, hi=1024, Hq=14, Hkv=2, D=64, train=True),
        # one sample through one layer of a log-probability worker: the smallest attention call
        _attn("attn_one_sample", tokens=777, lo=777, hi=777, Hq=12, Hkv=2, D=128, train=False),
        # log-probabilities, entropy and backward on logits a caller has materialised (a per-token function of its own)
        dict(kind="rows", name="rows_logits", dtype="bf16", rows=2048, V=151936),
        # the trainer's whole micro-batch from Python lists: packing, loss, metrics, gradients (0.5B-class head, prompts
        # masked)
        _host("trainer_micro_batch", kind="trainer", samples=16, H=896, V=151936, p_lo=32, p_hi=256, lo=128, hi=768),
        # the log-probability worker's whole batch from Python lists to the packed host result (0.5B-class head)
        _host("logprob_worker", kind="worker", samples=24, H=896, V=151936, p_lo=32, p_hi=256, lo=128, hi=768),
    ]


def _step(name, **kw):
    return dict(kind="step", name=name, **kw)


def _logprob(name, **kw):
    return dict(kind="logprob", name=name, **kw)


def _attn(name, **kw):
    return dict(kind="attn", name=name, **kw)


def _host(name, **kw):
    return dict(name=name, **kw)


_HEADS = ((896, 151936), (1536, 151936), (3584, 152064), (5120, 152064), (8192, 128256))
_ATTN_HEADS = ((12, 2, 128), (28, 4, 128), (16, 4, 128), (14, 2, 64), (32, 8, 64))


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("step", "step", "step", "fp32", "logprob", "attn", "attn", "attn", "rows", "trainer", "worker"))
    most = 6.0 * 35871 * 3584 * 152064                       # the largest listed case
    if kind == "step":
        H, V = rng.choice(_HEADS)
        tokens = _log_int(rng, 200, min(36000, int(most / (6.0 * H * V))))
        kl = rng.choice((0.0, 0.001, 0.04))
        hi = min(tokens, rng.choice((1024, 2048, 8192)))
        return dict(kind="step", dtype="bf16", tokens=tokens, H=H, V=V, lo=min(128, hi), hi=hi, kl=kl,
                    agg=rng.choice(("token_mean", "sample_mean")), chunk=rng.choice((0, 2048, 4096, 8192)))
    if kind == "fp32":
        tokens = _log_int(rng, 100, 2000)
        return dict(kind="step", dtype="fp32", tokens=tokens, H=rng.choice((64, 96, 128, 256)), V=_log_int(rng, 500, 8000),
                    lo=16, hi=64, kl=rng.choice((0.0, 0.001)), agg=rng.choice(("token_mean", "sample_mean")), chunk=0)
    if kind == "logprob":
        H, V = rng.choice(_HEADS)
        tokens = _log_int(rng, 200, min(48000, int(most / (2.0 * H * V))))
        hi = min(tokens, rng.choice((1024, 4096)))
        return dict(kind="logprob", tokens=tokens, H=H, V=V, lo=min(128, hi), hi=hi)
    if kind == "attn":
        Hq, Hkv, D = rng.choice(_ATTN_HEADS)
        tokens = _log_int(rng, 200, 36000)
        hi = min(tokens, rng.choice((512, 1024, 2048, 8192)))
        return dict(kind="attn", tokens=tokens, lo=min(128, hi), hi=hi, Hq=Hq, Hkv=Hkv, D=D, train=rng.random() < 0.75)
    if kind == "rows":
        dtype = rng.choice(("bf16", "bf16", "fp32"))
        return dict(kind="rows", dtype=dtype, rows=_log_int(rng, 128, 3000), V=rng.choice((151936, 152064, 128256, 32001)))
    H, V = rng.choice(_HEADS[:2])
    return dict(kind=kind, samples=_log_int(rng, 2, 40), H=H, V=V, p_lo=16, p_hi=_log_int(rng, 32, 512), lo=128,
                hi=_log_int(rng, 256, 1024))


# ------------------------------------------------------------------------------------------------ inputs
def _lengths(case):
    """Sample lengths that add up to the case's tokens; a matter of the case alone, so that every seed has the same
    work (the seed deals their order)."""
    rng = random.Random(case["tokens"] * 31 + case["hi"])
    out, total = [], 0
    while total < case["tokens"]:
        k = case["lo"] if case["lo"] == case["hi"] else _log_int(rng, case["lo"], case["hi"]) if case["hi"] > 1024 \
            else rng.randint(case["lo"], case["hi"])
        k = min(k, case["tokens"] - total)
        if k < 2 and out:                                    # one token alone has nothing to score
            out[-1] += k
        else:
            out.append(k)
        total += k
    return out


def _dtype(case):
    return torch.float32 if case.get("dtype") == "fp32" else torch.bfloat16


def _advantages(n, rng):
    """Group-normalised 0/1 rewards, one advantage per sample."""
    out = []
    while len(out) < n:
        r = np.array([float(rng.random() < 0.5) for _ in range(GROUP)])
        out.extend(((r - r.mean()) / (r.std() + 1e-4)).tolist())
    return out[:n]


def _head(H, V, dtype, gen):
    return (torch.randn(V, H, generator=gen, device="cuda", dtype=torch.float32) * 0.02).to(dtype)


def _packed(lens, V, gen):
    """Token ids, labels (each sample's first token is its prompt) and segment boundaries of one packed row."""
    T = sum(lens)
    ids = torch.randint(0, V, (T,), generator=gen, device="cuda")
    cu = torch.tensor([0] + np.cumsum(lens).tolist(), dtype=torch.int32, device="cuda")
    labels = ids.clone()
    labels[cu[:-1].long()] = IGNORE
    return labels.view(1, T), cu


def _policy_hidden(weight, labels, gen):
    """Final hidden states of a policy that could have written the tokens: unit-variance noise plus a push towards
    the next token's row of the head, its logit raised by 2..16."""
    T, (V, H) = labels.numel(), weight.shape
    y = torch.nn.functional.pad(labels.view(-1), (0, 1), value=0)[1:].clamp(min=0)
    h = torch.randn(T, H, generator=gen, device="cuda", dtype=torch.float32)
    push = (torch.rand(T, 1, generator=gen, device="cuda") * 14 + 2) / (0.02 * 0.02 * H)
    for a in range(0, T, 4096):
        h[a:a + 4096] += weight[y[a:a + 4096]].float() * push[a:a + 4096]
    return h.to(weight.dtype).view(1, T, H)


def _rollout_logprobs(hidden, weight, labels, gen):
    """What the sampling engine reported: log-probabilities of logits in the weights' type, a little off-policy."""
    h = hidden.view(-1, hidden.shape[-1])
    y = torch.nn.functional.pad(labels.view(-1), (0, 1), value=IGNORE)[1:]
    lp = torch.empty(h.shape[0], device="cuda")
    for a in range(0, h.shape[0], 2048):
        x = torch.matmul(h[a:a + 2048], weight.t())
        t = x.gather(1, y[a:a + 2048].clamp(min=0).view(-1, 1)).view(-1).float()
        lp[a:a + 2048] = t - torch.logsumexp(x.float(), dim=1)
    lp += torch.randn(lp.shape, generator=gen, device="cuda") * 0.05
    return torch.where(y == IGNORE, torch.zeros_like(lp), lp)


class _Body(torch.nn.Module):
    """Stand-in for the transformer body: a frozen embedding and one trainable layer."""

    def __init__(self, V, H):
        super().__init__()
        self.embed_tokens = torch.nn.Embedding(V, H)
        self.embed_tokens.weight.requires_grad_(False)
        self.proj = torch.nn.Linear(H, H, bias=False)

    def forward(self, input_ids=None, position_ids=None, **kw):
        return (self.proj(self.embed_tokens(input_ids)),)


class _Config:
    output_attentions = False
    output_hidden_states = False
    use_return_dict = True


class _Policy(torch.nn.Module):
    def __init__(self, V, H, gen):
        super().__init__()
        with torch.device("meta"):
            self.model = _Body(V, H)
            self.lm_head = torch.nn.Linear(H, V, bias=False)
        self.to_empty(device="cuda")
        self.to(torch.bfloat16)
        with torch.no_grad():
            self.lm_head.weight.copy_(_head(H, V, torch.bfloat16, gen))
            self.model.embed_tokens.weight.copy_(_head(H, V, torch.bfloat16, gen) * 50)
            self.model.proj.weight.copy_(torch.randn(H, H, generator=gen, device="cuda") / math.sqrt(H))
        self.config = _Config()


class _TrainConfig:
    clip_low, clip_high, clip_ratio_c = 0.2, 0.28, 3.0
    entropy_coeff = 0.0

    def __init__(self, samples):
        self.train_minibatch_sample_size = samples


def _samples(case, seed):
    """Rollouts as the reference's controller holds them: Python lists per sample."""
    sizes = random.Random(case["samples"] * 31 + case["hi"])
    lens = [(sizes.randint(case["p_lo"], case["p_hi"]), sizes.randint(case["lo"], case["hi"])) for _ in range(case["samples"])]
    rng = random.Random(seed)
    rng.shuffle(lens)
    values = np.random.default_rng(seed)
    adv = _advantages(len(lens), rng)
    out = []
    for i, (li, lo) in enumerate(lens):
        ids = values.integers(0, case["V"], li + lo)
        out.append(dict(sample_ids=ids.tolist(), sample_position_ids=list(range(li + lo)),
                        labels=[IGNORE] * li + ids[li:].tolist(), input_len=li, output_len=lo, advantage=adv[i],
                        reward=float(adv[i] > 0), modified_reward=None, delimiter_not_found=False, truncated_sample=False))
    return out


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    if kind in ("step", "logprob", "attn"):
        lens = _lengths(case)
        random.Random(seed).shuffle(lens)
    if kind in ("step", "logprob"):
        weight = _head(case["H"], case["V"], _dtype(case), gen)
        labels, cu = _packed(lens, case["V"], gen)
        hidden = _policy_hidden(weight, labels, gen)
        state = dict(kind=kind, hidden=hidden, weight=weight, labels=labels)
        if kind == "step":
            old = _rollout_logprobs(hidden, weight, labels, gen)
            adv = torch.repeat_interleave(torch.tensor(_advantages(len(lens), random.Random(seed)), device="cuda"),
                                          torch.tensor(lens, device="cuda")).float()
            args = dict(temperature=1.0, old_logprobs=old, advantages=adv, clip_low=0.2, clip_high=0.28, clip_ratio_c=3.0,
                        loss_chunksize=case["chunk"] or None)
            if case["agg"] == "sample_mean":
                args.update(loss_agg_mode="sample_mean", cu_seqlens=cu)
            if case["kl"]:
                ref = old + torch.randn(old.shape, generator=gen, device="cuda") * 0.05
                args.update(ref_logprobs=ref, kl_beta=case["kl"])
            state.update(args=args)
            hidden.requires_grad_(True)
            weight.requires_grad_(True)
        return state
    if kind == "attn":
        T, D = case["tokens"], case["D"]
        cu = torch.tensor([0] + np.cumsum(lens).tolist(), dtype=torch.int32, device="cuda")
        q, k, v, dout = (torch.randn(T, n, D, generator=gen, device="cuda").to(torch.bfloat16).requires_grad_(case["train"])
                         for n in (case["Hq"], case["Hkv"], case["Hkv"], case["Hq"]))
        return dict(kind=kind, q=q, k=k, v=v, cu=cu, longest=max(lens), dout=dout.detach(), train=case["train"])
    if kind == "rows":
        N, V = case["rows"], case["V"]
        labels = torch.randint(0, V, (N,), generator=gen, device="cuda")
        logits = torch.empty(N, V, device="cuda", dtype=_dtype(case))
        for a in range(0, N, 512):
            logits[a:a + 512] = torch.randn(min(512, N - a), V, generator=gen, device="cuda")
        logits[torch.arange(N, device="cuda"), labels] += 10
        labels[torch.rand(N, generator=gen, device="cuda") < 0.1] = IGNORE
        g = torch.randn(N, generator=gen, device="cuda").to(logits.dtype) / N
        return dict(kind=kind, logits=logits.requires_grad_(True), labels=labels, g=g)
    model = _Policy(case["V"], case["H"], gen)
    samples = _samples(case, seed)
    if kind == "worker":
        G.make_grpo_forward(model, mode="eval")
        return dict(kind=kind, harness=W.LogProbHarness(model), samples=samples)
    with torch.no_grad():                                    # the sampling engine's log-probabilities, as lists
        for s in samples:
            ids = torch.tensor(s["sample_ids"], device="cuda").view(1, -1)
            labels = torch.tensor(s["labels"], device="cuda").view(1, -1)
            lp = _rollout_logprobs(model.model(input_ids=ids)[0], model.lm_head.weight, labels, gen)
            s["sample_logprobs"] = lp.tolist()
            s["sample_entropies"] = [11.0] * len(s["sample_ids"])
    G.make_grpo_forward(model, mode="training", loss_chunksize=4096)
    return dict(kind=kind, harness=W.TrainerHarness(model, _TrainConfig(case["samples"])), samples=samples, model=model)


# ------------------------------------------------------------------------------------------------ one pass
def run(state):
    kind = state["kind"]
    if kind == "step":
        out = G.grpo_loss_and_entropy_ce_fn(state["weight"], None, state["hidden"], state["labels"], **state["args"])
        grads = torch.autograd.grad(out[0], (state["hidden"], state["weight"]))
        return tuple(t.detach() for t in out) + grads
    if kind == "logprob":
        with torch.no_grad():
            return G.fused_log_probs_and_entropy_fn(state["weight"], None, state["hidden"], state["labels"], 1.0)
    if kind == "attn":
        q, k, v, cu = state["q"], state["k"], state["v"], state["cu"]
        if not state["train"]:
            with torch.no_grad():
                return flash_attn_varlen_func(q, k, v, cu, cu, state["longest"], state["longest"], causal=True)
        out = flash_attn_varlen_func(q, k, v, cu, cu, state["longest"], state["longest"], causal=True)
        return (out.detach(),) + torch.autograd.grad(out, (q, k, v), state["dout"])
    if kind == "rows":
        lp = G.logprobs_from_logits(state["logits"], state["labels"])
        ent = G.entropy_from_logits(state["logits"])
        return (lp.detach(), ent) + torch.autograd.grad(lp, state["logits"], state["g"])
    if kind == "worker":
        return state["harness"].compute_log_probs_from_samples(state["samples"], packed=True).buffer
    model = state["model"]
    model.zero_grad(set_to_none=True)
    metrics = state["harness"].compute_gradients(state["samples"])
    return dict(metrics, grad_head=model.lm_head.weight.grad, grad_proj=model.model.proj.weight.grad)


# ------------------------------------------------------------------------------------------------ what it takes
def work(case):
    kind = case["kind"]
    if kind == "rows":
        size = 4 if case["dtype"] == "fp32" else 2
        return dict(bytes=2.0 * case["rows"] * case["V"] * size, flops=8.0 * case["rows"] * case["V"])
    if kind == "attn":
        pairs = sum(n * (n + 1) // 2 for n in _lengths(case))
        row = case["tokens"] * case["D"] * 2.0
        q, kv = row * case["Hq"], row * case["Hkv"]
        bytes_ = 2 * q + 2 * kv + (2 * q + 2 * kv if case["train"] else 0)
        return dict(bytes=bytes_, flops=(14.0 if case["train"] else 4.0) * pairs * case["D"] * case["Hq"])
    size = 4 if case.get("dtype") == "fp32" else 2
    H, V = case["H"], case["V"]
    if kind in ("step", "logprob"):
        T = scored = case["tokens"]
    else:
        sizes = random.Random(case["samples"] * 31 + case["hi"])
        lens = [(sizes.randint(case["p_lo"], case["p_hi"]), sizes.randint(case["lo"], case["hi"])) for _ in range(case["samples"])]
        T, scored = sum(a + b for a, b in lens), sum(b for _, b in lens)
    operands = (float(T) * H + float(V) * H) * size
    if kind in ("logprob", "worker"):
        return dict(bytes=operands + 16.0 * T, flops=2.0 * scored * H * V)
    return dict(bytes=2 * operands + 40.0 * T, flops=6.0 * scored * H * V)


def tolerance(case):
    """About four times what the outputs differ from the same quantities in 64 bits, or formed by the package's other
    route to them (logits recomputed in the backward)."""
    if case["kind"] == "step" and case["dtype"] == "fp32":
        return dict(rel=2e-4)            # the log ratio, a small difference of log-probabilities, at 5e-5; gradients 6e-6
    if case["kind"] in ("logprob", "worker"):
        return dict(rel=3e-5)            # fp32 sums over bf16 operands: 6e-6
    if case["kind"] == "rows":
        return dict(rel=1e-5 if case["dtype"] == "fp32" else 7e-3)
    return dict(rel=1e-2)                # bf16 gradients and attention outputs: 2e-3 .. 4e-3
