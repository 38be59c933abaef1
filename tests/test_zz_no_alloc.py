"""The allocation-free entry point of the C ABI, ``lf_launch_decode_static``: a split decode
step whose split-K partials live in a static device array of the library.  Its output must be
bit-equal to the step through ``lf_launch`` with a caller-owned scratch buffer (same kernels,
same partials), on two calls in a row, the second with a smaller input; a step whose partials
exceed the array is refused before anything is launched."""
import pytest
import torch

from loopfuse_amd import lowering, runtime, workloads

pytestmark = pytest.mark.gpu


def _step(w, splits, **kw):
    plan = lowering.AttnPlan(scale=w.scale, k_paged=w.k_table is not None, v_paged=w.v_table is not None)
    return lowering.attention(w.q, w.k, w.v, plan, w.k_table, w.v_table, num_splits=splits, **kw)


def test_static_scratch_decode_matches_caller_owned_scratch():
    dev = torch.device("cuda:0")
    first = True
    for name, B, S, splits in (("c5", 16, 2048, 4), ("c5", 4, 512, 2), ("c4", 2, 1024, 4)):
        w = workloads.make(name, seed=7, B=B, S=S).to(dev)
        want = _step(w, splits).clone()
        assert lowering.attention.last_launch["kernels"] == ["lf_attn_decode", "lf_attn_decode_combine"]
        got = torch.full_like(want, float("nan"))
        torch.cuda.synchronize()
        allocs = torch.cuda.memory_stats()["allocation.all.allocated"]
        _step(w, splits, out=got, static_scratch=True)
        assert lowering.attention.last_launch.get("static_scratch") is True
        if not first:       # the first call may load the code object; later calls allocate nothing at all
            assert torch.cuda.memory_stats()["allocation.all.allocated"] == allocs
        first = False
        torch.cuda.synchronize()
        assert torch.equal(got, want), (name, B, S, splits)


def test_static_scratch_refuses_oversized_steps():
    dev = torch.device("cuda:0")
    w = workloads.make("c5", seed=7, B=64, S=2048).to(dev)
    out = torch.empty_like(w.q)
    need = 64 * 8 * 4 * 16 * (128 + 2) * 4
    assert need > runtime.static_scratch_bytes()
    with pytest.raises(runtime.ShimError) as e:
        _step(w, 16, out=out, static_scratch=True)
    assert e.value.code == -4 and "static scratch" in str(e.value)
    # and an unsplit step is not what this entry point is for
    with pytest.raises(lowering.UnsupportedPlan):
        _step(w, 1, out=out, static_scratch=True)


@pytest.mark.parametrize("B,Hq,Hkv,S,page", [(96, 16, 16, 1024, 16), (16, 64, 8, 8192, 1)])
def test_static_scratch_chooses_splits_that_fit(B, Hq, Hkv, S, page):
    """No count given: a step that would run unsplit, and one whose partials would not fit."""
    g = torch.Generator(device="cuda").manual_seed(B)
    q = torch.randn((B, Hq, 1, 128), generator=g, device="cuda").bfloat16()
    shape = (B * S // page, page, Hkv, 128) if page > 1 else (B * S, Hkv, 128)
    k, v = (torch.randn(shape, generator=g, device="cuda").bfloat16() for _ in range(2))
    table = torch.randperm(B * S // page, generator=g, device="cuda").view(B, S // page).int()
    plan = lowering.AttnPlan(scale=128 ** -0.5, k_paged=True, v_paged=True)
    out = torch.empty_like(q)
    lowering.attention(q, k, v, plan, table, table, out=out, static_scratch=True)
    splits = lowering.attention.last_launch["grid"][1]
    assert splits > 1 and torch.equal(out, lowering.attention(q, k, v, plan, table, table, num_splits=splits))


def test_captured_split_steps_keep_their_scratch():
    """A split decode step captured into a graph, then a larger one on the same stream (which replaces the buffer that calls
    on a stream share) and other tensors in the memory that is free afterwards: every replay gives the eager result and
    leaves those tensors alone."""
    w, big = (workloads.make("c5", seed=7, B=B, S=2048).to(torch.device("cuda")) for B in (2, 24))
    want, want_big = _step(w, 4).clone(), _step(big, 16).clone()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        _step(w, 4)                      # the shared buffer of this stream
    torch.cuda.synchronize()
    g, g_big = torch.cuda.CUDAGraph(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        got = _step(w, 4)
    with torch.cuda.stream(s):
        _step(big, 16)
    with torch.cuda.graph(g_big, stream=s):
        got_big = _step(big, 16)
    others = [torch.full((1 << 20,), 3.0, device="cuda") for _ in range(8)]
    for _ in range(3):
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)
        g_big.replay()
        torch.cuda.synchronize()
        assert torch.equal(got_big, want_big) and all(bool((t == 3.0).all()) for t in others)
