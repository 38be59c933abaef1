"""Launches repeated from the record of a call with the same signature (``lowering._Kept``)."""
import os

import pytest
import torch

import loopfuse_amd  # noqa: F401
from loopfuse_amd import lowering
from loopfuse_amd.lowering import AttnPlan, attention, attention_backward

BF = torch.bfloat16


def _fresh(fn):
    """``fn()`` through the general path, and what it recorded."""
    lowering._kept.clear()
    return fn(), dict(lowering._last_launch._get())


def test_no_signature_for_what_is_not_plain(monkeypatch):
    """Tensors that are not on the GPU, a plan that holds a tensor, options that are no plain values and an environment put in
    the place of the imported one leave a call to the general path."""
    q = torch.zeros((1, 1, 1, 64), dtype=BF)
    assert lowering._signature("fwd", (q, None), AttnPlan(), None) is None
    assert lowering._signature("fwd", (None,), AttnPlan(scale=torch.tensor(1.0)), None) is None
    assert lowering._signature("fwd", (None,), AttnPlan(), {"bn": torch.tensor(32)}) is None
    monkeypatch.setattr(os, "environ", dict(os.environ))
    assert lowering._signature("fwd", (None,), AttnPlan(), None) is None


def _r(shape, seed, dtype=BF):
    return torch.randn(shape, generator=torch.Generator(device="cuda").manual_seed(seed), device="cuda").to(dtype)


def _paged(seed, page, B=2, Hkv=8, S=512, D=128):
    n = S // page
    pool = (B * n, Hkv, D) if page == 1 else (B * n, page, Hkv, D)
    table = torch.randperm(B * n, generator=torch.Generator(device="cuda").manual_seed(seed), device="cuda").view(B, n).to(torch.int32)
    return _r(pool, seed), _r(pool, seed + 1), table


FORMS = {
    "prefill": lambda s: ((_r((2, 4, 300, 128), s), _r((2, 2, 300, 128), s + 1), _r((2, 2, 300, 128), s + 2), AttnPlan("causal", scale=0.1)), {}),
    "prefill views": lambda s: ((_r((2, 300, 4, 64), s).transpose(1, 2), _r((2, 300, 4, 64), s + 1).transpose(1, 2),
                                 _r((2, 300, 4, 64), s + 2).transpose(1, 2), AttnPlan("sliding", window=50, scale=0.1, softcap=20.0)), {}),
    "prefill into a view": lambda s: ((_r((2, 4, 100, 64), s), _r((2, 4, 100, 64), s + 1), _r((2, 4, 100, 64), s + 2), AttnPlan(scale=0.1)),
                                      {"out": torch.zeros((2, 100, 4, 64), dtype=BF, device="cuda").transpose(1, 2)}),
    "prefill with lse": lambda s: ((_r((1, 4, 100, 64), s), _r((1, 4, 100, 64), s + 1), _r((1, 4, 100, 64), s + 2), AttnPlan("causal", scale=0.1)),
                                   {"lse": torch.zeros((1, 4, 100), device="cuda"), "choice": {"prefill": "swp"}}),
    "decode": lambda s: ((_r((3, 8, 1, 64), s), _r((3, 2, 700, 64), s + 1), _r((3, 2, 700, 64), s + 2), AttnPlan(scale=0.1)), {}),
    "decode paged": lambda s: ((_r((2, 16, 1, 128), s), *_paged(s, 16)[:2], AttnPlan(scale=0.1, k_paged=True, v_paged=True), *[_paged(s, 16)[2]] * 2), {}),
    "decode one-token pages, whole": lambda s: ((_r((2, 8, 1, 128), s), *_paged(s, 1)[:2], AttnPlan(scale=0.1, k_paged=True, v_paged=True),
                                                 *[_paged(s, 1)[2]] * 2), {"choice": {"splits": 1}}),
    "padded head dim": lambda s: ((_r((2, 2, 60, 40), s), _r((2, 2, 60, 40), s + 1), _r((2, 2, 60, 40), s + 2), AttnPlan(scale=0.1)), {}),
}


@pytest.mark.gpu
@pytest.mark.parametrize("form", list(FORMS), ids=lambda f: f.replace(" ", "_"))
def test_a_repeated_call_is_the_general_path_on_its_own_tensors(form):
    """Every form of call: the bits and the record of launches of the general path, for tensors that were not there when the launches
    were recorded, whose results and log-sum-exps are written and no earlier call's; replayed from a graph as well."""
    args, kw = FORMS[form](1)
    attention(*args, **kw)                                    # recorded
    for seed in (11, 12):
        args, kw = FORMS[form](seed)
        before = len(lowering._kept)
        got, lse = attention(*args, **kw), kw.get("lse")
        assert len(lowering._kept) == before and before       # repeated
        record = dict(lowering._last_launch._get())
        lse = None if lse is None else lse.clone()
        mine = got.clone()
        want, full = _fresh(lambda: attention(*args, **kw))
        assert torch.equal(mine, want) and record == full
        assert lse is None or torch.equal(lse, kw["lse"])
        assert "out" not in kw or got is kw["out"]
    graph, out = torch.cuda.CUDAGraph(), None
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        out = attention(*args, **kw)
    for _ in range(3):
        out.zero_()
        graph.replay()
        attention(*FORMS[form](21)[0], **kw if "choice" in kw and "lse" not in kw else {})
        torch.cuda.synchronize()
        assert torch.equal(out, mine) and ("out" not in kw or out is kw["out"])


@pytest.mark.gpu
def test_what_changes_the_launches_changes_the_signature(monkeypatch):
    """A switch set after the launches were recorded, another option, other strides, another length: each takes the route it would
    take in a new process; a refusal is not recorded, and a call that is refused is refused again."""
    def call(S=512, view=False, **kw):
        q, k, v = (_r((1, 4, S, 64), i) for i in range(3))
        if view:
            k = _r((1, S, 4, 64), 1).transpose(1, 2)
        return attention(q, k, v, AttnPlan("causal", scale=0.1), **kw)

    lowering._kept.clear()
    base = call()
    assert lowering._last_launch["kernels"] == ["lf_attn_prefill_swp"] and len(lowering._kept) == 1
    call(choice={"prefill": "w32"})
    assert lowering._last_launch["kernels"] == ["lf_attn_prefill"]
    monkeypatch.setenv("LOOPFUSE_PREFILL", "w32")
    call()
    assert lowering._last_launch["kernels"] == ["lf_attn_prefill"]
    monkeypatch.delenv("LOOPFUSE_PREFILL")
    assert torch.equal(call(), base) and lowering._last_launch["kernels"] == ["lf_attn_prefill_swp"]
    call(S=500)
    call(view=True)
    assert len(lowering._kept) == 5
    q, k = _r((1, 4, 64, 64), 1), _r((1, 4, 64, 64), 2)
    for _ in range(2):
        with pytest.raises(lowering.UnsupportedPlan):
            attention(q, k, k.float(), AttnPlan(scale=0.1))
        with pytest.raises(lowering.UnsupportedPlan):
            attention(q, k, k, AttnPlan(scale=float("nan")))
    assert len(lowering._kept) == 5


@pytest.mark.gpu
@pytest.mark.parametrize("D,mask,keep", [(128, "causal", None), (64, None, False), (128, "sliding", True)])
def test_a_repeated_backward_is_the_general_path(D, mask, keep):
    def operands(seed):
        q, k, v, dout = _r((2, 4, 200, D), seed), _r((2, 2, 200, D), seed + 1), _r((2, 2, 200, D), seed + 2), _r((2, 4, 200, D), seed + 3)
        lse = torch.empty((2, 4, 200), device="cuda")
        o = attention(q, k, v, plan, lse=lse, choice={"prefill": "swp"})
        return q, k, v, o, lse, dout, plan

    plan = AttnPlan(mask, window=70 if mask == "sliding" else 0, scale=0.1)
    attention_backward(*operands(1), keep_ds=keep)
    args = operands(31)
    before = len(lowering._kept)
    got = attention_backward(*args, keep_ds=keep)
    record = dict(lowering._last_launch._get())
    assert len(lowering._kept) == before
    want, full = _fresh(lambda: attention_backward(*args, keep_ds=keep))
    assert all(torch.equal(a, b) for a, b in zip(got, want)) and record == full


@pytest.mark.gpu
def test_a_dispatch_mode_still_sees_the_training_ops(monkeypatch):
    """A training graph calls its attention past the dispatcher, except where something is there that has to see the ops."""
    import functools

    from torch.utils._python_dispatch import TorchDispatchMode

    from loopfuse_amd import loopfuse_backend
    from loopfuse_amd.torch_backend import training

    class Seen(TorchDispatchMode):
        def __init__(self):
            super().__init__()
            self.names = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.names.append(str(func))
            return func(*args, **(kwargs or {}))

    def attn(q, k, v):
        s = torch.ops.loopfuse.causal_mask(q @ k.transpose(-2, -1) * 0.125)
        return torch.softmax(s, dim=-1) @ v

    graphs, direct_calls = [], training.direct_calls
    monkeypatch.setattr(training, "direct_calls", lambda gm: (graphs.append(direct_calls(gm)), graphs[-1])[1])
    fn = torch.compile(attn, backend=functools.partial(loopfuse_backend, mode=None), dynamic=False)
    q, k, v = (_r((1, 2, 100, 64), i).requires_grad_(True) for i in range(3))
    dout = _r((1, 2, 100, 64), 9)
    out = fn(q, k, v)
    want = torch.autograd.grad(out, (q, k, v), dout)
    before = dict(training.counters)
    inner = fn(q, k, v)
    got = torch.autograd.grad(inner, (q, k, v), dout)
    assert training.counters["fwd"] == before["fwd"] + 1 and training.counters["bwd"] == before["bwd"] + 1
    assert torch.equal(inner, out) and all(torch.equal(a, b) for a, b in zip(got, want))
    targets = [n.target for gm in graphs for n in gm.graph.nodes if n.op == "call_function"]
    assert all(targets.count(call) == 1 and op not in targets for op, call in training._DIRECT.items())
    mode = Seen()
    call = training._DIRECT[torch.ops.loopfuse_amd.attention_fwd.default]
    with torch.no_grad(), mode:
        call(q.detach(), k.detach(), v.detach(), 1, 0, 0.125, 0.0)
    assert any("attention_fwd" in n for n in mode.names)


def test_only_plain_tensors_pass_the_dispatcher():
    """A view whose negation is still to be applied, a tensor whose gradient is recorded and a subclass, in the place of any
    operand, go through the op."""
    from loopfuse_amd.torch_backend import training

    class Sub(torch.Tensor):
        pass

    call = training._direct(lambda *a: "op", lambda *a: "direct", 3)
    a = torch.zeros(2, 4)
    assert call(a, a, a, 1) == "direct" and call(a, torch.nn.Parameter(a, requires_grad=False), a, 1) == "direct"
    neg = torch.zeros(2, 4, dtype=torch.complex64).conj().imag
    grad = torch.zeros(2, 4, requires_grad=True)
    for odd in (neg, grad, a.as_subclass(Sub)):
        for at in range(3):
            assert call(*[odd if i == at else a for i in range(3)], 1) == "op"
    with torch.no_grad():
        assert call(grad, grad, grad, 1) == "direct"


def _record_of_a_backward(ds_shape):
    """A record of ``attention_backward`` whose launches only count, and operands on the CPU for it."""
    class Launches:
        count = 0

        def launch(self, params):
            self.count += 1

    kept = lowering._Kept.__new__(lowering._Kept)
    kept.params, kept.launches = bytes(lowering.AttnBwdParams()), Launches()
    kept.results, kept.scratch, kept.record, kept.calls = (BF, ds_shape), None, {"kernels": []}, None
    q, k = torch.zeros((1, 4, 40, 64), dtype=BF), torch.zeros((1, 2, 40, 64), dtype=BF)
    return kept, (q, k, k, q, torch.zeros((1, 4, 40)), q)


def _no_room_for(monkeypatch, shape):
    """``torch.empty`` finds no room for tensors of ``shape``; returns the list of the shapes that it is asked for."""
    asked, empty = [], torch.empty

    def limited(size, *args, **kw):
        asked.append(tuple(size))
        if tuple(size) == shape:
            raise torch.OutOfMemoryError("no room")
        return empty(size, *args, **kw)

    monkeypatch.setattr(torch, "empty", limited)
    return asked


def test_a_repeated_backward_takes_its_results_before_ds(monkeypatch):
    """The results and delta are what a call needs, dS is what it can do without: allocated last, so that it cannot take their
    room, and where it finds none nothing is launched and the caller is told."""
    shape = (4, 3, lowering.BWD_DS_BLOCK)
    kept, args = _record_of_a_backward(shape)
    asked = _no_room_for(monkeypatch, shape)
    assert lowering._backward_again(kept, *args) is None and kept.launches.count == 0
    assert asked == [(1, 4, 40, 64), (1, 2, 40, 64), (1, 2, 40, 64), (1, 4, 40), shape]
    monkeypatch.undo()
    dq, dk, dv = lowering._backward_again(kept, *args)
    assert kept.launches.count == 1 and dq.shape == args[0].shape and dk.shape == dv.shape == args[1].shape


@pytest.mark.gpu
@pytest.mark.parametrize("recorded", [False, True])
def test_a_backward_without_room_for_ds_looks_for_it_once(recorded, monkeypatch):
    """No room on the first call of a signature, or on a repeated one that had it: the gradients of the form without dS, which is
    what the following calls repeat without another attempt, until many calls later there is room again."""
    q, k, v, dout = (_r((2, h, 300, 128), i) for i, h in enumerate((4, 2, 2, 4)))
    plan, lse = AttnPlan("causal", scale=0.1), torch.empty((2, 4, 300), device="cuda")
    args = (q, k, v, attention(q, k, v, plan, lse=lse, choice={"prefill": "swp"}), lse, dout, plan)
    shape = (8, lowering.bwd_ds_blocks(lowering.MASK_CAUSAL, 0, 300, 300), lowering.BWD_DS_BLOCK)
    assert lowering.bwd_keep_ds(128, False, 8, 2, 300, 8 * shape[1])
    want = attention_backward(*args, keep_ds=False)
    lowering._kept.clear()
    monkeypatch.setattr(lowering, "_NO_ROOM_CALLS", 3)
    with_ds = None
    for _ in range(3 if recorded else 0):
        with_ds = attention_backward(*args)
    asked = _no_room_for(monkeypatch, shape)
    for attempts in (1, 1, 1, 1, 2):
        got = attention_backward(*args)
        assert all(torch.equal(a, b) for a, b in zip(got, want)) and asked.count(shape) == attempts
    with pytest.raises(torch.OutOfMemoryError):
        attention_backward(*args, keep_ds=True)
    monkeypatch.undo()
    lowering._kept.clear()
    got = attention_backward(*args)
    assert lowering._last_launch["kernels"] == ["lf_attn_bwd_delta", "lf_attn_bwd_dkdv", "lf_attn_bwd_dq"]
    assert with_ds is None or all(torch.equal(a, b) for a, b in zip(got, with_ds))


@pytest.mark.gpu
def test_a_recorded_call_launches_through_its_record(monkeypatch):
    """The first call of a signature too: one call of the library for all its kernels."""
    from loopfuse_amd import runtime

    calls = []
    one, many = runtime.Kernel.launch, runtime.LaunchList.launch
    monkeypatch.setattr(runtime.Kernel, "launch", lambda self, *a, **kw: (calls.append("one"), one(self, *a, **kw))[1])
    monkeypatch.setattr(runtime.LaunchList, "launch", lambda self, *a: (calls.append("list"), many(self, *a))[1])
    for form in ("prefill", "decode", "decode paged"):
        args, kw = FORMS[form](41)
        lowering._kept.clear()
        calls.clear()
        first, second = attention(*args, **kw), attention(*args, **kw)
        assert calls == ["list", "list"] and torch.equal(first, second)


def test_a_specialisation_hashes_anew_in_another_process():
    """The hash is formed once per object, and is not what a copy in another process, whose strings hash otherwise, may keep."""
    import dataclasses
    import pickle

    spec = lowering.bwd_spec(BF, 64, lowering.MASK_CAUSAL)
    assert hash(spec) == hash(dataclasses.replace(spec)) and spec.__dict__["_hash"] == hash(spec)
    again = pickle.loads(pickle.dumps(spec))
    assert "_hash" not in again.__dict__ and again == spec and {spec: 1}[again] == 1
    assert dataclasses.replace(spec, head_dim=128) != spec and hash(dataclasses.replace(spec, head_dim=128)) != hash(spec)


def test_a_tuned_choice_is_not_taken_from_before_the_kernels_changed(monkeypatch, tmp_path):
    """The file of measured choices holds those of other kernels and rules too: they are neither found nor written again."""
    import json

    q, k = torch.zeros((1, 8, 1, 64), dtype=BF), torch.zeros((1, 8, 500, 64), dtype=BF)
    key = lowering._tune_key(q, k, AttnPlan(scale=0.1), None, 0)
    path = tmp_path / "autotune.json"
    monkeypatch.setattr(lowering, "_TUNE_FILE", str(path))
    monkeypatch.setattr(lowering, "_tuned", {})
    path.write_text(json.dumps({key: {"splits": 4}, key.rsplit("|r", 1)[0]: {"splits": 2}, key[:-1] + "x": {"splits": 8}}))
    lowering._load_tuned()
    assert lowering._tuned == {key: {"splits": 4}}
    monkeypatch.setattr(lowering, "_rules_version", lambda: "later")
    assert lowering._tune_key(q, k, AttnPlan(scale=0.1), None, 0) != key
    lowering._tuned.clear()
    lowering._load_tuned()
    assert lowering._tuned == {}
