"""Host-side logic that needs no GPU: numpy forms of the batch-shaping helpers
against the oracle, synthetic workload generators, and the refusal of CPU
tensors by the product path."""
import warnings

import numpy as np
import pytest
import torch

from oracle import grpo_oracle as O


def test_numpy_index_and_broadcast_helpers_match_oracle():
    import sample_processing_utils as spu
    rng = np.random.default_rng(1)
    for n in (0, 1, 7):
        il = rng.integers(1, 9, n)
        ol = rng.integers(0, 9, n)
        assert np.array_equal(spu.get_output_logits_indices_numba(il, ol), O.output_logits_indices(il, ol))
        vals = rng.normal(size=n)
        assert np.array_equal(spu.broadcast_values(vals, il + ol), O.broadcast_values(vals, il + ol))


def test_product_path_refuses_cpu_tensors():
    import grpo_loss as G
    hs = torch.randn(1, 8, 16)
    W = torch.randn(32, 16)
    labels = torch.randint(0, 32, (1, 8))
    with pytest.raises(RuntimeError, match="GPU"):
        G.fused_log_probs_and_entropy_fn(W, None, hs, labels)
    with pytest.raises(RuntimeError, match="GPU"):
        G.grpo_loss_and_entropy_ce_fn(W, None, hs, labels, advantages=torch.zeros(8))
    with pytest.raises(RuntimeError, match="GPU"):
        G.logprobs_from_logits(torch.randn(4, 9), torch.zeros(4, dtype=torch.long))


def test_fused_step_refuses_a_zero_temperature():
    """Its reciprocal would be infinite; the refusal comes before any tensor is looked at."""
    from fgrpo import ops
    h, w, y = torch.randn(4, 64), torch.randn(10, 64), torch.zeros(4, dtype=torch.long)
    with pytest.raises(ZeroDivisionError):
        ops.fused_grpo_loss(h, w, None, y, torch.zeros(4), torch.zeros(4), temperature=0.0)


def test_foreign_per_token_fn_needs_the_gpu_too():
    """A caller-supplied per_token_fn takes the materialised-logits route; that route has no CPU version either."""
    import grpo_loss as G
    with pytest.raises(RuntimeError, match="GPU"):
        G.fused_log_probs_and_entropy_fn(torch.randn(4, 4), None, torch.randn(1, 2, 4), torch.zeros(1, 2, dtype=torch.long),
                                         per_token_fn=lambda *a, **k: None)


def test_reference_surface_is_present():
    import grpo_loss as G
    import inspect
    for name in ("GRPOOutput", "LogProbsOutput", "make_grpo_forward", "logprobs_from_logits",
                 "logprobs_from_logits_flash_attn", "entropy_from_logits", "fused_log_probs_and_entropy_fn",
                 "ce_loss_and_entropy_logsoftmax", "grpo_loss_and_entropy_ce_fn",
                 "grpo_loss_and_entropy_ce_from_logsoftmax", "compute_dual_clip_grpo_loss", "COMPUTE_ENTROPY_FN",
                 "DEBUG", "debug_print"):
        assert hasattr(G, name), name
    sig = inspect.signature(G.grpo_loss_and_entropy_ce_fn)
    assert list(sig.parameters) == ["lm_head_weights", "lm_head_bias", "hidden_states", "labels", "temperature",
                                    "old_logprobs", "advantages", "clip_low", "clip_high", "clip_ratio_c",
                                    "ce_loss_and_entropy_fn", "per_token_fn", "loss_chunksize", "unused_kwargs"]
    d = {k: v.default for k, v in sig.parameters.items()}
    assert (d["temperature"], d["clip_low"], d["clip_high"], d["clip_ratio_c"], d["loss_chunksize"]) == (1.0, 0.2, 0.4, 1e32, None)
    sig = inspect.signature(G.compute_dual_clip_grpo_loss)
    assert list(sig.parameters) == ["policy_model", "minibatch", "clip_low", "clip_high", "clip_ratio_c",
                                    "compute_entropy", "apply_entropy_bonus", "entropy_coeff"]
    sig = inspect.signature(G.make_grpo_forward)
    assert list(sig.parameters) == ["model", "temperature", "mode", "use_torch_compile", "loss_chunksize"]


def test_synthetic_workloads_have_the_stated_shapes():
    from fgrpo.synthetic import make_workload, CONFIGS
    w = make_workload("cfg0")
    assert w.H == 64 and w.V == 1000 and w.n_samples == 16 and 16 * 16 <= w.T <= 16 * 64
    assert w.hidden.shape == (1, w.T, 64) and w.weight.shape == (1000, 64) and w.dtype == torch.float32
    assert int(w.cu_seqlens[-1]) == w.T and w.cu_seqlens.dtype == torch.int32
    assert (w.labels[0, w.cu_seqlens[:-1].long()] == -100).all()
    assert (w.labels != -100).sum() == w.T - w.n_samples
    assert torch.equal(O.cu_seqlens_from_position_ids(w.position_ids), w.cu_seqlens)
    w2 = make_workload("cfg0")
    assert torch.equal(w.hidden, w2.hidden) and torch.equal(w.labels, w2.labels)
    # a shrunken cfg1: same generator code path, exact token count
    w1 = make_workload("cfg1", overrides=dict(H=64, V=512, tokens=4096))
    assert w1.T == 4096 and w1.dtype == torch.bfloat16 and int(w1.cu_seqlens[-1]) == 4096
    assert min(w1.sample_lens) >= 2
    assert set(CONFIGS) == {"cfg0", "cfg1", "cfg2", "cfg3", "cfg4"}


def test_varlen_attention_argument_errors_and_route():
    """Unsupported flash-attn options raise before anything touches the GPU; a model switched to the varlen
    attention reaches the HIP op (which refuses CPU tensors: there is no fallback)."""
    import torch
    import varlen_attention as VA
    q = torch.zeros(8, 2, 128, dtype=torch.bfloat16)
    cu = torch.tensor([0, 8], dtype=torch.int32)
    with pytest.raises(RuntimeError, match="dropout"):
        VA.flash_attn_varlen_func(q, q, q, cu, cu, 8, 8, dropout_p=0.1)
    with pytest.raises(RuntimeError, match="window_size"):
        VA.flash_attn_varlen_func(q, q, q, cu, cu, 8, 8, window_size=(128, 0))
    with pytest.raises(RuntimeError, match="share their segments"):
        VA.flash_attn_varlen_func(q, q, q, cu, torch.tensor([0, 4, 8], dtype=torch.int32), 8, 8)
    with pytest.raises(RuntimeError, match="GPU"):
        VA.flash_attn_varlen_func(q, q, q, cu, cu, 8, 8, causal=True)
    from transformers import Qwen2Config, Qwen2ForCausalLM
    cfg = Qwen2Config(vocab_size=64, hidden_size=256, intermediate_size=256, num_hidden_layers=1,
                      num_attention_heads=2, num_key_value_heads=1, max_position_embeddings=64)
    model = Qwen2ForCausalLM(cfg)
    assert VA.install_explicit_varlen_wrapper(model) is True
    with pytest.raises(RuntimeError, match="GPU"):
        model(input_ids=torch.zeros(1, 6, dtype=torch.long), position_ids=torch.tensor([[0, 1, 2, 0, 1, 2]]))


def test_missing_library_raises_and_nothing_falls_back(monkeypatch, tmp_path):
    """Without libfgrpo.so the product raises (naming the build command) instead of computing some other way."""
    from fgrpo import _lib
    monkeypatch.setattr(_lib, "LIB_PATH", str(tmp_path / "no_such_libfgrpo.so"))
    monkeypatch.setattr(_lib, "_lib", None)              # forget the handle loaded by earlier tests
    with pytest.raises(RuntimeError, match="fgrpo.build"):
        _lib.load()
    import grpo_loss as G
    import torch
    with pytest.raises(RuntimeError):                    # the drop-in has no other way to compute
        G.logprobs_from_logits(torch.zeros(2, 8), torch.zeros(2, dtype=torch.long))


def test_product_modules_never_import_the_oracle():
    """The oracle is test infrastructure: no module of the package imports, reads or names it."""
    import os
    root = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "async-grpo-nccl_amd")
    for dirpath, _, files in os.walk(root):
        for f in files:
            if f.endswith((".py", ".h", ".hip")):
                text = open(os.path.join(dirpath, f), encoding="utf-8").read()
                assert "oracle" not in text, os.path.join(dirpath, f)


def test_packed_logprobs_container():
    """The wire format of the logprob worker's result on the host side: validation, views, list form."""
    import sample_processing_utils as spu
    buf = torch.arange(12, dtype=torch.float32).reshape(2, 6)
    p = spu.PackedLogProbs(buf, [0, 2, 2, 6])
    assert len(p) == 3 and p.has_entropies and p.offsets.dtype == np.int32
    lp, ent = p.sample(2)
    assert lp.tolist() == [2.0, 3.0, 4.0, 5.0] and ent.tolist() == [8.0, 9.0, 10.0, 11.0]
    assert np.shares_memory(lp, buf.numpy())
    assert p.to_lists() == [{"logprobs": [0.0, 1.0], "entropies": [6.0, 7.0]}, {"logprobs": [], "entropies": []},
                            {"logprobs": [2.0, 3.0, 4.0, 5.0], "entropies": [8.0, 9.0, 10.0, 11.0]}]
    only_lp = spu.PackedLogProbs(buf[:1], [0, 6])
    assert not only_lp.has_entropies and only_lp.to_lists() == [{"logprobs": [0.0, 1.0, 2.0, 3.0, 4.0, 5.0], "entropies": None}]
    samples = [{}, {}, {}]
    p.attach(samples)
    assert spu._packed_run(samples) == (p, 0, 3) and spu._packed_run(samples[1:]) == (p, 1, 3)
    assert spu._packed_run([samples[2], samples[0]]) is None and spu._packed_run([{}]) is None
    for bad in ([0, 7], [1, 6], [0, 4, 3, 6]):
        with pytest.raises(ValueError):
            spu.PackedLogProbs(buf, bad)
    with pytest.raises(ValueError):
        spu.PackedLogProbs(buf.double(), [0, 6])
    with pytest.raises(ValueError):
        p.attach([{}])


def test_host_addresses_are_not_handed_to_kernels():
    from fgrpo import ops
    assert ops._ptr(None) is None
    with pytest.raises(RuntimeError, match="must live on the GPU"):
        ops._ptr(torch.zeros(4))


def test_the_list_of_scored_rows_goes_to_forwards_that_take_it():
    import functools
    from types import SimpleNamespace
    from workers import _takes_row_list

    def made(input_ids=None, labels=None, **unused):
        return None
    made.takes_compact_masked_tokens = True

    @functools.wraps(made)
    def wide(*args, **kwargs):
        return made(*args, **kwargs)

    @functools.wraps(made)
    def narrow(input_ids, labels):
        return made(input_ids=input_ids, labels=labels)

    class Own(torch.nn.Module):
        def forward(self, input_ids, labels):
            return input_ids + labels

    traced = torch.jit.trace(Own(), (torch.zeros(1), torch.zeros(1)))
    inner = SimpleNamespace(forward=made)
    assert _takes_row_list(inner) and _takes_row_list(SimpleNamespace(forward=wide))
    assert _takes_row_list(SimpleNamespace(forward=lambda **kw: None, module=inner))
    for model in (Own(), traced, SimpleNamespace(forward=narrow), SimpleNamespace(forward=narrow, module=inner),
                  SimpleNamespace(forward=lambda **kw: None), SimpleNamespace(forward=lambda **kw: None, module=traced), lambda **kw: None):
        assert not _takes_row_list(model)


def test_what_a_forward_takes_is_read_as_its_signature_says():
    import functools
    import inspect
    from workers import _takes_keyword

    class Call:
        def __call__(self, a, *, rows=None):
            return a

        def method(self, rows):
            return rows

        @classmethod
        def made(cls, **kw):
            return kw

        @staticmethod
        def free(a, *args):
            return a

    def local_only(a):
        rows = a
        return rows

    def two(a, rows):
        return a, rows
    for f in (Call(), Call().method, Call.made, Call.free, local_only, two, lambda a, rows=1: a, lambda rows, /: rows,
              functools.partial(two, 1), functools.partial(local_only), Call().__call__):
        params = inspect.signature(f, follow_wrapped=False).parameters.values()
        want = any(p.kind is p.VAR_KEYWORD or (p.name == "rows" and p.kind is not p.POSITIONAL_ONLY) for p in params)
        assert _takes_keyword(f, "rows") == want
    assert not _takes_keyword(None, "rows") and not _takes_keyword(torch.jit.script(torch.nn.Linear(2, 2)).forward, "rows")


class _Int(int):
    pass


@pytest.mark.parametrize("dtype", [np.int64, np.float32])
@pytest.mark.parametrize("items", [
    [], [7], list(range(-3, 900)), (1, 2, 3), [2 ** 63 - 1, -2 ** 63], [2 ** 63], [True, 2], [_Int(5), 6], [np.int64(9), 1],
    [1.0, 2.5, -0.0], [0.1] * 700, [float("nan"), float("inf"), -float("inf")], [3.5e38], [1e-45, 1e-50], [np.float32(0.5), 1.0],
    [1, 2.0], [None], ["4"], [1, None]])
def test_packed_lists_are_what_numpy_makes_of_them(dtype, items):
    """Every form of entry, those that are read natively and those that are not: the same values, or the same error."""
    from sample_processing_utils import _fill

    def outcome(write):
        dst = np.full(len(items) + 2, 77, dtype=dtype)
        try:
            write(dst[1:-1])
        except (TypeError, ValueError, OverflowError) as e:
            return type(e)
        assert dst[0] == 77 and dst[-1] == 77
        return dst.tobytes()

    def by_numpy(piece):
        piece[:] = np.fromiter(items, dtype=dtype, count=len(items))
    with np.errstate(all="ignore"):
        assert outcome(lambda piece: _fill(piece, [{"x": items}], "x", [len(items)])) == outcome(by_numpy)


def test_packed_lists_of_several_samples_follow_each_other():
    from sample_processing_utils import _fill
    dst = np.zeros(9, dtype=np.int64)
    _fill(dst, [{"x": [1, 2]}, {}, {"x": (np.int32(3),)}, {"x": torch.tensor([4, 5])}, {"x": []}, {"x": (6, 7)}], "x",
          [2, 2, 1, 2, 0, 2], default=-100)
    assert dst.tolist() == [1, 2, -100, -100, 3, 4, 5, 6, 7]
    with pytest.raises(ValueError):
        _fill(dst, [{"x": [1, 2]}], "x", [3])


@pytest.mark.parametrize("missing", ["BINDING_PATH", "LIB_PATH"])
def test_packing_needs_no_extension_module(monkeypatch, tmp_path, missing):
    """Where the library or the extension module is not built, packing works as before there was one."""
    from fgrpo import _lib
    from sample_processing_utils import _fill
    monkeypatch.setattr(_lib, missing, str(tmp_path / "not_built.so"))
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "_native", None)
    with pytest.raises(RuntimeError, match="fgrpo.build"):
        _lib.native()
    dst = np.zeros(8, dtype=np.int64)
    _fill(dst, [{"x": np.array([1, 2])}, {"x": torch.tensor([3])}, {"x": [4, 5]}, {"x": (6,)}, {}], "x", [2, 1, 2, 1, 2], default=-100)
    assert dst.tolist() == [1, 2, 3, 4, 5, 6, -100, -100]


@pytest.fixture(scope="module")
def attn_route(tmp_path_factory):
    """csrc/attn_route.h, which is plain C++, behind three C functions."""
    import ctypes as C
    import os
    import subprocess
    where = tmp_path_factory.mktemp("attn_route")
    src, lib = str(where / "route.cpp"), str(where / "route.so")
    with open(src, "w") as f:
        f.write('#include "attn_route.h"\nextern "C" {\nusing ll = long long;\n'
                "int reach(ll st, int rows, int D) { return fgrpo::attn_rows_in_reach(st, rows, D); }\n"
                "int query(int w, ll q, ll k, ll v, int Hq, int D) { return fgrpo::attn_query_form(w, q, k, v, Hq, D); }\n"
                "int key(int w, ll q, ll k, ll v, int T, int Hq, int Hkv, int D, int keys) {"
                " return fgrpo::attn_key_form(w, q, k, v, T, Hq, Hkv, D, keys); }\n}\n")
    csrc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "async-grpo-nccl_amd", "csrc")
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-O1", "-fPIC", "-shared", f"-I{csrc}", src, "-o", lib], check=True)
    lib = C.CDLL(lib)
    lib.reach.argtypes = [C.c_longlong, C.c_int, C.c_int]
    lib.query.argtypes = [C.c_int] + [C.c_longlong] * 3 + [C.c_int] * 2
    lib.key.argtypes = [C.c_int] + [C.c_longlong] * 3 + [C.c_int] * 5
    return lib


def _last_stride(rows, D):
    """Largest multiple of eight elements at which the last byte of `rows` rows is within 32-bit offsets of the first row."""
    st = (2 ** 32) // (2 * (rows - 1)) // 8 * 8
    while (rows - 1) * st * 2 + 2 * D > 2 ** 32 - 1:
        st -= 8
    return st


@pytest.mark.parametrize("rows", [32, 64])
@pytest.mark.parametrize("D", [64, 128])
def test_attention_rows_are_in_reach_up_to_the_last_byte(attn_route, rows, D):
    last = _last_stride(rows, D)
    for st in (8, 3584, last - 8, last):
        assert attn_route.reach(st, rows, D) and (rows - 1) * st * 2 + 2 * D < 2 ** 32
    for st in (last + 8, 2 * last, 2 ** 40, 2 ** 62):
        assert not attn_route.reach(st, rows, D) and (rows - 1) * st * 2 + 2 * D >= 2 ** 32


@pytest.mark.parametrize("D,keys", [(64, 32), (128, 64)])
def test_attention_rows_out_of_reach_take_the_64_bit_kernels(attn_route, D, keys):
    """Each stride by itself on both sides of each kernel's reach: 32 rows of Q, 64 of K and V for the query side; 32 of Q and
    `keys` of K and V, or 64 of Q, for dK/dV."""
    row, at32, at64 = 2 * D, _last_stride(32, D), _last_stride(64, D)
    for wanted in (0, 1, 2, 3):
        form = lambda q=row, k=row, v=row, Hq=4: attn_route.query(wanted, q, k, v, Hq, D)
        for near in (dict(), dict(q=at64 + 8), dict(q=at32), dict(k=at64), dict(v=at64), dict(Hq=at32 // D)):
            assert form(**near) == wanted, near
        for far in (dict(q=at32 + 8), dict(k=at64 + 8), dict(v=at64 + 8), dict(k=2 ** 50), dict(Hq=at32 // D + 1)):
            assert form(**far) == 1, far
    at = _last_stride(keys, D)
    form = lambda w=0, q=row, k=row, v=row, T=1000, Hq=4, Hkv=2: attn_route.key(w, q, k, v, T, Hq, Hkv, D, keys)
    for near in (dict(), dict(q=at32), dict(k=at), dict(v=at), dict(w=3)):
        assert form(**near) == 3, near
    for mid in (dict(k=at + 8), dict(v=at + 8), dict(k=2 ** 50, q=at64), dict(w=2), dict(w=2, k=2 ** 40, q=at64),
                dict(T=2 ** 28), dict(T=2 ** 28 - 1, Hq=8, Hkv=1)):
        assert form(**mid) == 2, mid
    for far in (dict(q=at32 + 8), dict(k=at + 8, q=at64 + 8), dict(w=2, q=at64 + 8), dict(w=1), dict(w=2, T=2 ** 28, q=at32 + 8),
                dict(Hq=at32 // D + 1, Hkv=1)):
        assert form(**far) == 1, far


@pytest.mark.parametrize("form", [list, tuple, np.array, torch.tensor, lambda x: [torch.tensor(v) for v in x],
                                  lambda x: np.array(x, dtype=np.int32), lambda x: torch.tensor(x, dtype=torch.int32).view(2, 2)])
def test_output_indices_take_lengths_in_any_host_form(monkeypatch, form):
    """What the kernel is handed, read back as the kernel reads it: n offsets, n input lengths, n + 1 output offsets."""
    import contextlib
    import ctypes
    import types
    from fgrpo import ops
    il, ol = [3, 1, 4, 2], [2, 5, 1, 0]

    def kernel(tok, lin, out, n, total, dst, stream):
        at = lambda p, k, t: np.ctypeslib.as_array((t * k).from_address(p))
        tok, lin, out = at(tok, n, ctypes.c_int32), at(lin, n, ctypes.c_int32), at(out, n + 1, ctypes.c_int32)
        for i in range(n):
            at(dst, total, ctypes.c_int64)[out[i]:out[i + 1]] = tok[i] + lin[i] - 1 + np.arange(out[i + 1] - out[i])
        return 0

    monkeypatch.setattr(ops._lib, "load", lambda: types.SimpleNamespace(fgrpo_output_indices=kernel))
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    monkeypatch.setattr(ops, "_ptr", lambda t: t.data_ptr())
    monkeypatch.setattr(torch.cuda, "device", lambda d: contextlib.nullcontext())
    got = ops.output_indices(form(il), form(ol), torch.device("cpu"))
    assert got.tolist() == O.output_logits_indices(il, ol).tolist()


@pytest.mark.parametrize("il,ol", [([3, 4, 5], [2]), ([3], [2]), ([1] * 9, [3] * 9), ([], []), ([], [4])])
def test_output_indices_pack_holds_what_the_kernel_reads(il, ol):
    """3 n + 1 entries for n samples, also where one output length is given for all: the kernel reads n + 1 output offsets."""
    from fgrpo import ops
    n = len(il)
    a, b = torch.tensor(il, dtype=torch.int64), torch.tensor(ol, dtype=torch.int64)
    tok, out = torch.zeros(n, dtype=torch.int64), torch.zeros(n + 1, dtype=torch.int64)
    tok[1:], out[1:] = torch.cumsum(a + b, 0)[:-1], torch.cumsum(b, 0)
    assert ops.output_indices_pack(il, ol).tolist() == torch.cat([tok, a, out]).tolist()


@pytest.mark.parametrize("il,ol", [([3, 4, 5], [2, 1]), ([3], [2, 1]), ([3, 4], []), ([3, 4, 5], [0, 0])])
def test_output_indices_refuse_other_numbers_of_lengths(monkeypatch, il, ol):
    from fgrpo import ops
    monkeypatch.setattr(ops._lib, "load", lambda: None)
    for call in (ops.output_indices_pack, lambda *a: ops.output_indices(*a, torch.device("cpu"))):
        with pytest.raises(RuntimeError):
            call(il, ol)


@pytest.mark.parametrize("H,T,narrow", [(4096, 832, 0.5), (4608, 776, 0.5), (4608, 777, 0.6), (5120, 832, 0.6), (6144, 832, 0.6),
                                        (8192, 832, 0.5), (1536, 832, 0.5), (5120, 896, 0.65)])
def test_shares_of_a_narrow_last_token_tile(H, T, narrow):
    """594 vocabulary tiles in 66 shares of nine for three whole token tiles; the narrow one's shares take as long.  Seen in
    the workspace, which holds 16 bytes a token and share (with 256 CUs, which is also what a host without a GPU plans for)."""
    from fgrpo import _lib
    V, up = 152064, lambda n: (n + 255) // 256 * 256
    shares = -(-594 // int(9 / narrow))
    want = up(16 * 66 * T) + up(16 * shares * (T % 256)) + up(4 * T) + up(4 * V)
    assert _lib.load().fgrpo_logprob_fwd_workspace(T, H, V, _lib.BF16) == want


@pytest.mark.parametrize("replaced", [False, True])
def test_the_trainer_calls_the_loss_its_module_names(monkeypatch, replaced):
    """``workers.compute_dual_clip_grpo_loss`` is the loss of ``grpo_loss``, and what a program puts in its place is what the
    trainer calls; otherwise the metrics are read behind the backward."""
    import grpo_loss
    import workers
    assert workers.compute_dual_clip_grpo_loss is grpo_loss.compute_dual_clip_grpo_loss
    seen, x = [], torch.ones(3, requires_grad=True)
    batch = {"_num_output_tokens_non_masked_host": 3.0}
    monkeypatch.setattr(workers, "post_process_batch", lambda samples, device: batch)

    def loss_of(model, minibatch, clip_low, clip_high, clip_ratio_c, **kw):
        assert minibatch is batch and (clip_low, clip_high, clip_ratio_c) == (0.2, 0.28, 3.0)
        assert kw == dict(compute_entropy=True, apply_entropy_bonus=True, entropy_coeff=0.0)
        seen.append("loss")
        return (x * x).sum()

    def read():
        seen.append("metrics behind" if x.grad is not None else "metrics before")
        return {"loss": 3.0}
    if replaced:
        monkeypatch.setattr(workers, "compute_dual_clip_grpo_loss", lambda *a, **kw: (loss_of(*a, **kw), read()))
    else:
        monkeypatch.setattr(workers, "dual_clip_grpo_loss_begin", lambda *a, **kw: (loss_of(*a, **kw), read))
    harness = workers.TrainerHarness(torch.nn.Linear(1, 1), device="cpu")
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")                       # autocast for a device that is not there
        assert harness.compute_gradients([{}]) == {"loss": 3.0}
    assert seen == ["loss", "metrics before" if replaced else "metrics behind"]
    assert torch.equal(x.grad, 2 * x.detach())
