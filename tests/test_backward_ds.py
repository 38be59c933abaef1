"""dS left in memory by ``lf_attn_bwd_dkdv`` and read by ``lf_attn_bwd_dq`` (``lowering.bwd_keep_ds``), and the split of
a tile's queries over the waves of ``lf_attn_bwd_dkdv`` (``lowering.bwd_q_split``)."""
import pytest
import torch

from loopfuse_amd import lowering
from loopfuse_amd.lowering import AttnPlan, attention, attention_backward

MASKS = {None: lowering.MASK_NONE, "causal": lowering.MASK_CAUSAL, "sliding": lowering.MASK_SLIDING}


def _row(mask, qb, nkb, window):
    """``lf_bw_ds_row`` of csrc/kernels/lf_attn_bwd.hip."""
    if mask is None:
        return qb * nkb
    if mask == "causal":
        m = min(qb, nkb)
        return m * (m + 1) // 2 + (qb - m) * nkb
    before = (window + 30) // 32
    return qb * (before + 1) - (qb - before)


@pytest.mark.parametrize("mask,window", [(None, 0), ("causal", 0), ("sliding", 1), ("sliding", 2), ("sliding", 33), ("sliding", 64), ("sliding", 1000)])
def test_blocks_of_ds_have_places_of_their_own(mask, window):
    """Every 32 x 32 block that holds a visible score has a place inside the head's scratch, no two the same, and a row of
    blocks lies in the order of its keys (what the loads of lf_attn_bwd_dq rely on)."""
    for Sq in (1, 31, 32, 33, 200, 417):
        for Sk in (1, 32, 65, 200, 530):
            nqb, nkb = -(-Sq // 32), -(-Sk // 32)
            total = lowering.bwd_ds_blocks(MASKS[mask], window, Sq, Sk)
            seen = set()
            for qb in range(nqb):
                for kb in range(nkb):
                    q0, k0, k1 = 32 * qb, 32 * kb, min(32 * kb + 32, Sk) - 1
                    if (mask is None) or (k0 <= q0 and (mask == "causal" or q0 - k1 < window)):
                        at = _row(mask, qb, nkb, window) + kb
                        assert 0 <= at < total and at not in seen
                        seen.add(at)


def _plan(D, mask, window, cap):
    return AttnPlan(mask=mask, window=window, scale=D ** -0.5, softcap=cap)


CASES = [  # B, Hq, Hkv, Sq, Sk, D, mask, window, softcap
    (2, 4, 2, 300, 300, 128, "causal", 0, None), (1, 4, 1, 517, 200, 128, "causal", 0, None), (1, 2, 2, 200, 517, 64, "causal", 0, None),
    (2, 4, 2, 300, 333, 64, None, 0, None), (1, 1, 1, 1, 65, 128, None, 0, None), (1, 2, 2, 96, 31, 128, None, 0, None),
    (1, 4, 4, 700, 700, 128, "sliding", 100, None), (2, 2, 1, 600, 600, 64, "sliding", 1, None), (1, 2, 1, 333, 333, 64, "causal", 0, 30.0),
    (1, 2, 2, 400, 400, 128, "sliding", 5000, 30.0), (1, 2, 2, 257, 129, 128, "sliding", 33, None)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_gradients_from_the_kept_ds(case, dtype):
    """Tails of both sequences, grouped heads, the three masks, a softcap, both splits of both kernels: dK and dV have the bits
    of the launch that keeps nothing (same delta launch), dQ is as close to it as the rounding of dS to the operand type leaves
    two orders of the same sums, and repeats have the same bits."""
    B, Hq, Hkv, Sq, Sk, D, mask, window, cap = case
    g = torch.Generator(device="cuda").manual_seed(1)
    q, dout = (torch.randn((B, Hq, Sq, D), generator=g, device="cuda").to(dtype) for _ in range(2))
    k, v = (torch.randn((B, Hkv, Sk, D), generator=g, device="cuda").to(dtype) for _ in range(2))
    plan = _plan(D, mask, window, cap)
    lse = torch.empty((B, Hq, Sq), device="cuda")
    o = attention(q, k, v, plan, lse=lse, choice={"prefill": "swp"})
    seen = torch.isfinite(o).all(dim=-1)                  # rows that see no key have no gradient to compare
    o = torch.where(seen[..., None], o, 0)
    lse = torch.where(seen, lse, float("inf"))            # P = 0 there
    for blocks in (1, 2) if lowering.bwd_two_key_blocks(D, MASKS[mask], cap is not None) else (1,):
        for threads in (256, 512):
            kw = dict(key_blocks=blocks, dq_threads=threads, q_split=False)
            kept = attention_backward(q, k, v, o, lse, dout, plan, keep_ds=True, **kw)
            assert lowering._last_launch["kernels"] == ["lf_attn_bwd_delta", "lf_attn_bwd_dkdv", "lf_attn_bwd_dq"]
            again = attention_backward(q, k, v, o, lse, dout, plan, keep_ds=True, **kw)
            plain = attention_backward(q, k, v, o, lse, dout, plan, keep_ds=False, **{**kw, "dq_threads": 512})
            assert all(torch.equal(a, b) for a, b in zip(kept, again))
            assert torch.equal(kept[1], plain[1]) and torch.equal(kept[2], plain[2])
            a, b = kept[0].double(), plain[0].double()
            assert torch.isfinite(a).all()
            # either is within one unit of rounding of dS (2^-8 / 2^-11 of each term, at random) and of the result of the exact sum
            assert (a - b).norm() <= (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11) * b.norm() + 1e-6 * dout.double().norm()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_queries_of_a_tile_split_over_the_waves(case, dtype):
    """The same cases with the queries of a tile split: tails in either half of a tile, a last tile whose second half is empty,
    keys that fill one wave of a workgroup only.  dK and dV are fp32 sums in another order (two of half as many terms) of the same
    rounded P and dS, rounded once: within a few last bits of a result here and there; dQ from the kept dS has the bits it has
    without the split, and repeats have the same bits."""
    B, Hq, Hkv, Sq, Sk, D, mask, window, cap = case
    g = torch.Generator(device="cuda").manual_seed(3)
    q, dout = (torch.randn((B, Hq, Sq, D), generator=g, device="cuda").to(dtype) for _ in range(2))
    k, v = (torch.randn((B, Hkv, Sk, D), generator=g, device="cuda").to(dtype) for _ in range(2))
    plan = _plan(D, mask, window, cap)
    lse = torch.empty((B, Hq, Sq), device="cuda")
    o = attention(q, k, v, plan, lse=lse, choice={"prefill": "swp"})
    seen = torch.isfinite(o).all(dim=-1)
    o = torch.where(seen[..., None], o, 0)
    lse = torch.where(seen, lse, float("inf"))
    for keep in (False, True):
        kw = dict(keep_ds=keep, key_blocks=1, dq_threads=512)
        split = attention_backward(q, k, v, o, lse, dout, plan, q_split=True, **kw)
        again = attention_backward(q, k, v, o, lse, dout, plan, q_split=True, **kw)
        whole = attention_backward(q, k, v, o, lse, dout, plan, q_split=False, **kw)
        assert all(torch.equal(a, b) for a, b in zip(split, again))
        assert torch.equal(split[0], whole[0])
        # fp32 sums of up to Sq * group terms differ by 2^-24 sqrt(terms) of the terms' size; 1e-6 is 16 x that.  A result that
        # then rounds the other way moves by one unit in the last place of 8 / 11 significant bits: 2^-7 / 2^-10 of itself at most
        for a, b in zip(split[1:], whole[1:]):
            assert torch.isfinite(a).all()
            eps = 2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -10
            assert ((a.double() - b.double()).abs() <= eps * b.double().abs() + 1e-6 * dout.double().norm()).all()
            assert (a != b).double().mean() < 0.02
    with pytest.raises(lowering.UnsupportedPlan):
        attention_backward(q, k, v, o, lse, dout, plan, key_blocks=2, q_split=True)
