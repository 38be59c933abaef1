"""dS left in memory by ``lf_attn_bwd_dkdv`` and read by ``lf_attn_bwd_dq`` (``lowering.bwd_keep_ds``)."""
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
            kw = dict(key_blocks=blocks, dq_threads=threads)
            kept = attention_backward(q, k, v, o, lse, dout, plan, keep_ds=True, **kw)
            assert lowering._last_launch["kernels"] == ["lf_attn_bwd_delta", "lf_attn_bwd_dkdv", "lf_attn_bwd_dq"]
            again = attention_backward(q, k, v, o, lse, dout, plan, keep_ds=True, **kw)
            plain = attention_backward(q, k, v, o, lse, dout, plan, keep_ds=False, key_blocks=blocks, dq_threads=512)
            assert all(torch.equal(a, b) for a, b in zip(kept, again))
            assert torch.equal(kept[1], plain[1]) and torch.equal(kept[2], plain[2])
            a, b = kept[0].double(), plain[0].double()
            assert torch.isfinite(a).all()
            # either is within one unit of rounding of dS (2^-8 / 2^-11 of each term, at random) and of the result of the exact sum
            assert (a - b).norm() <= (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11) * b.norm() + 1e-6 * dout.double().norm()
