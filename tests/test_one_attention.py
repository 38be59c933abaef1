"""Graphs that are one attention over their inputs: calls over plain tensors go past AOTAutograd's wrappers
(``training.one_attention``, ``interface._one_attention``), with their results and what they refuse."""
import functools

import pytest
import torch

from loopfuse_amd import loopfuse_backend
from loopfuse_amd.torch_backend import capture, interface, training


def _graph(second_output=False, extra=False, twice=False, perm=(0, 1, 2, 3), held=""):
    graph = torch.fx.Graph()
    ins = [graph.get_attr("_" + n) if n in held else graph.placeholder(n) for n in "qkv"]
    attr = graph.get_attr("_m")
    out = graph.call_function(training.fused_call_train, (attr, *((ins[0], ins[0], ins[2]) if twice else ins)))
    if extra:
        out = graph.call_function(torch.neg, (out,))
    graph.output((out, ins[0]) if second_output else (out,))
    ops = [capture.Operand(i, perm) for i in range(3)]
    root = torch.nn.Module()
    for n in held:
        setattr(root, "_" + n, torch.nn.Parameter(torch.zeros(1, 2, 8, 64, dtype=torch.bfloat16)))
    root._m = capture.AttentionMatch(out_node=None, inputs=ins, q=ops[0], k=ops[1], v=ops[2], factors=[0.125], post_factors=[],
                                     has_tanh=False, mask="causal", window=0, out_rank=4)
    return torch.fx.GraphModule(root, graph)


def test_only_graphs_of_one_attention_take_the_short_way():
    def general(*args):
        return "general"

    x = [torch.zeros(1, 2, 8, 64, dtype=torch.bfloat16) for _ in range(3)]
    assert training.one_attention(_graph(), x, general) is not general
    for other in (_graph(second_output=True), _graph(extra=True), _graph(twice=True), _graph(perm=(0, 2, 1, 3))):
        assert training.one_attention(other, x, general) is general
    # parameters and buffers that the graph holds itself (torch._dynamo.config.inline_inbuilt_nn_modules off)
    for held in ("k", "kv", "q"):
        assert training.one_attention(_graph(held=held), x[len(held):], general) is general
    assert training.one_attention(_graph(), [x[0], x[1], 7], general) is general
    assert training.one_attention(_graph(), [x[0][0], x[1][0], x[2][0]], general) is general
    # what is not plain is sent on, call by call
    call = training.one_attention(_graph(), x, general)
    assert call(*x) == "general"                     # the first one
    assert call(x[0], x[1], torch._neg_view(x[2])) == "general" and call(x[0], x[1]) == "general"

    class Sub(torch.Tensor):
        pass

    assert call(x[0].as_subclass(Sub), x[1], x[2]) == "general"


def _probabilities(q, k):
    return torch.softmax(torch.ops.loopfuse.causal_mask(q @ k.transpose(-2, -1) * (q.shape[-1] ** -0.5)), dim=-1)


def _alone(q, k, v, d):
    return torch.bmm(_probabilities(q, k), v)


def _out(q, k, v, d):
    torch.bmm(_probabilities(q, k), v, out=d)


def _out_returned(q, k, v, d):
    return torch.bmm(_probabilities(q, k), v, out=d)


def _copied(q, k, v, d):
    d.copy_(torch.bmm(_probabilities(q, k), v))


def _scaled_in_place(q, k, v, d):
    d.mul_(2.0)
    return torch.bmm(_probabilities(q, k), v)


def _input_returned(q, k, v, d):
    return torch.bmm(_probabilities(q, k), v), q


def _input_reshaped(q, k, v, d):
    d.unsqueeze_(0)
    return torch.bmm(_probabilities(q, k), v)


@pytest.mark.parametrize("refused", [False, True])
@pytest.mark.parametrize("fn", [_alone, _out, _out_returned, _copied, _scaled_in_place, _input_returned, _input_reshaped])
def test_what_the_short_way_leaves_in_outputs_and_inputs(fn, refused, monkeypatch):
    """Outputs and inputs after the first and the second call are those of the function itself, also where the kernels refuse the
    call (CPU tensors).  The graph that is nothing but an attention skips the general callable, one whose only result is
    written into an input does not, though it too is one attention with one output.  torch takes the kernel's place here."""
    short = []

    def run(self, vals):
        q, k, v = (self._operand(o, vals)[0] for o in (self.q, self.k, self.v))
        return (_probabilities(q, k) @ v)[0]

    real = interface._one_attention

    def seen(gm, found, general):
        short.append(real(gm, found, general) is not general)
        return real(gm, found, general)

    if not refused:
        monkeypatch.setattr(capture.AttentionMatch, "run", run)
    monkeypatch.setattr(interface, "_one_attention", seen)
    torch._dynamo.reset()
    compiled = torch.compile(fn, backend=functools.partial(loopfuse_backend, mode=None), dynamic=False)
    g = torch.Generator().manual_seed(1)
    for _ in range(2):
        want_in = [torch.randn(4, 40, 64, generator=g) for _ in range(4)]
        got_in = [t.clone() for t in want_in]
        with torch.no_grad():
            want, got = fn(*want_in), compiled(*got_in)
        torch.testing.assert_close(got, want)
        torch.testing.assert_close(got_in, want_in)
    if fn in (_alone, _out):
        assert short == [fn is _alone]


def _attn(q, k, v):
    s = torch.ops.loopfuse.causal_mask(q @ k.transpose(-2, -1) * (q.shape[-1] ** -0.5))
    return torch.softmax(s, dim=-1) @ v


def _compiled():
    torch._dynamo.reset()
    return torch.compile(_attn, backend=functools.partial(loopfuse_backend, mode=None), dynamic=False)


def _tensors(S=130):
    g = torch.Generator(device="cuda").manual_seed(S)
    return [torch.empty((2, 4, S, 64), dtype=torch.bfloat16, device="cuda").normal_(generator=g) for _ in range(4)]


@pytest.mark.gpu
@pytest.mark.parametrize("dout", ["dense", "strided", "expanded"])
def test_the_short_way_gives_the_bits_of_the_general_one(dout, monkeypatch):
    *x, d = _tensors()
    x = [t.requires_grad_() for t in x]
    d = {"dense": d, "strided": d.transpose(1, 2).contiguous().transpose(1, 2), "expanded": d[..., :1].expand_as(d)}[dout]

    def step(fn):
        out = fn(*x)
        return (out.detach(), *torch.autograd.grad(out, x, d))

    fn = _compiled()
    step(fn)
    before = dict(interface.stats)
    short = step(fn)
    assert interface.stats["fused_training"] == before["fused_training"] + 2
    assert torch.autograd.grad(fn(*x), x[1], d)[0].equal(short[2])
    with torch.no_grad():
        alone = fn(*x)
    assert interface.stats["fused"] == before["fused"] + 1
    monkeypatch.setattr(training, "one_attention", lambda gm, inputs, general: general)
    monkeypatch.setattr(interface, "_one_attention", lambda gm, found, general: general)
    fn = _compiled()
    assert all(a.equal(b) for a, b in zip(short, step(fn)))
    with torch.no_grad():
        assert fn(*x).equal(alone)


def _no_grad_values(q, k, v):
    with torch.no_grad():
        v = v * 0.5
    return _attn(q, k, v)


def _no_grad_angles(q, k, v):
    with torch.no_grad():      # (as rotary embeddings form theirs: nothing with a gradient is read)
        turn = torch.arange(q.shape[2], device=q.device).to(q.dtype)[:, None].cos()
    return _attn(q * turn, k, v)


_CUT = {"queries": lambda q, k, v: _attn(q.detach(), k, v), "data": lambda q, k, v: _attn(q, k.data, v), "values": _no_grad_values,
        "none": lambda q, k, v: _attn(q * 0.5, k, v), "nothing": _no_grad_angles}


@pytest.mark.parametrize("cut", sorted(_CUT))
def test_cut_gradients_are_seen(cut):
    seen = []
    torch._dynamo.reset()
    torch.compile(_CUT[cut], backend=lambda gm, inputs: (seen.append(interface._cuts_gradients(gm, inputs)), gm)[1])(
        *(torch.randn(1, 2, 8, 64, requires_grad=True) for _ in range(3)))
    assert seen == [cut in ("queries", "data", "values")]


@pytest.mark.gpu
@pytest.mark.parametrize("cut", sorted(_CUT))
def test_gradients_stop_where_the_function_stops_them(cut):
    *x, d = _tensors(70)
    x = [t.requires_grad_() for t in x]
    torch._dynamo.reset()
    fn = torch.compile(_CUT[cut], backend=functools.partial(loopfuse_backend, mode=None), dynamic=False)
    want = torch.autograd.grad(_CUT[cut](*x), x, d, allow_unused=True)
    graphs = interface.stats["training_graphs"]
    for _ in range(2):
        got = torch.autograd.grad(fn(*x), x, d, allow_unused=True)
        for a, w in zip(got, want):
            assert (a is None) == (w is None)
            # bf16 operands, probabilities and results on either side: 2^-9 each, a few of them per value
            assert a is None or ((a.double() - w.double()).norm() / w.double().norm()).item() <= 2e-2
    assert interface.stats["training_graphs"] == graphs + (cut in ("none", "nothing"))


def _counts(q, k, v, d, n):
    d.mul_(2.0)
    n += 1
    return _attn(q, k, v)


def test_a_trace_writes_to_copies():
    seen = []

    def backend(gm, inputs):
        names = [n.name for n in gm.graph.nodes if n.op == "placeholder"]
        seen.append({name.strip("l_"): a is not b for name, a, b in zip(names, inputs, interface._to_trace_on(gm, inputs))})
        return gm

    torch._dynamo.reset()
    leaf = [torch.randn(1, 2, 8, 64, requires_grad=True) for _ in range(4)]
    torch.compile(_counts, backend=backend)(*leaf[:3], leaf[3] * 1.0, torch.zeros(()))
    assert seen == [{"q": False, "k": False, "v": False, "d": True, "n": True}]


@pytest.mark.gpu
def test_the_first_call_writes_once():
    q, k, v, d = _tensors(60)
    q.requires_grad_()
    n, once = torch.zeros((), device="cuda"), 2.0 * d
    torch._dynamo.reset()
    fn = torch.compile(_counts, backend=functools.partial(loopfuse_backend, mode=None), dynamic=False)
    for calls in (1, 2):
        fn(q, k, v, d, n).sum().backward()
        assert n.item() == calls and torch.equal(d, once * 2.0 ** (calls - 1))


@pytest.mark.gpu
@pytest.mark.parametrize("buffer", [False, True])
def test_training_with_keys_that_the_graph_holds(buffer, monkeypatch):
    """Learnable keys and values of a module whose parameters are not inputs of its graph."""
    monkeypatch.setattr(torch._dynamo.config, "inline_inbuilt_nn_modules", False)
    q, k, v, d = _tensors(90)
    q.requires_grad_()

    class Memory(torch.nn.Module):
        def __init__(self):
            super().__init__()
            self.v = torch.nn.Parameter(v)
            if buffer:
                self.register_buffer("k", k)
            else:
                self.k = torch.nn.Parameter(k)

        def forward(self, q):
            return _attn(q, self.k, self.v)

    memory = Memory()
    torch._dynamo.reset()
    compiled = torch.compile(memory, backend=functools.partial(loopfuse_backend, mode=None), dynamic=False)
    given = [q, *memory.parameters()]
    want = torch.autograd.grad(_compiled()(q, memory.k, memory.v), given, d)
    before = interface.stats["fused_training"]
    for _ in range(2):
        got = torch.autograd.grad(compiled(q), given, d)
        assert all(a.equal(b) for a, b in zip(got, want))
    assert interface.stats["fused_training"] > before


@pytest.mark.gpu
def test_hooks_and_second_derivatives_of_the_short_way():
    *x, d = _tensors(100)
    x = [t.requires_grad_() for t in x]
    fn = _compiled()
    want = [torch.autograd.grad(fn(*x), x, d) for _ in range(2)][1]
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (packed.append(1), t.cpu())[1], lambda t: t.cuda()):
        out = fn(*x)
    assert len(packed) == 5 and all(a.equal(b) for a, b in zip(want, torch.autograd.grad(out, x, d)))
    first = torch.autograd.grad(fn(*x), x, d, create_graph=True)
    assert all(a.equal(b) for a, b in zip(want, first))
    with pytest.raises(RuntimeError):
        torch.autograd.grad(first[0].float().sum(), x[1])
