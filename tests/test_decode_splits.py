"""Work splits of decode steps: ``lowering.decode_even_split`` and the merge with one block per output row."""
import pytest
import torch

from loopfuse_amd import lowering
from loopfuse_amd.lowering import AttnPlan, attention


def test_even_splits_stay_within_their_limits():
    """64 splits at most, all but the last of the same length, 64 keys at least, the last what is left; the sequence is covered; a short sequence and a launch that fills the
    CUs by itself are left whole; a long one of few units is split over all CUs."""
    for D in (64, 128):
        for units in (1, 2, 8, 24, 96, 255, 256, 257, 700):
            for Sk in (16, 47, 96, 208, 1000, 8208, 65536):
                n = lowering.decode_even_split(units, Sk, D)
                splits, size = lowering._split_lengths(n, Sk)
                assert 1 <= splits <= n <= 64 and (splits == 1 or size >= 64) and 1 <= Sk - (splits - 1) * size <= size
        assert lowering.decode_even_split(256, 4000, D) == 1 and lowering.decode_even_split(4, 90, D) == 1
        assert lowering._split_lengths(lowering.decode_even_split(8, 20000, D), 20000)[0] >= 29
    for rows, nsplit in ((1, 1), (7, 4), (8, 5), (4097, 64)):
        for D in (64, 128):
            grid = lowering.decode_combine_grid(rows, nsplit, D)
            assert grid == rows or grid * (1024 // D) >= rows


@pytest.mark.parametrize("units,rows,Sk,D,splits", [
    # all counts measured: more splits cost the partials and the merge of many rows more than their shorter chains gain
    (32, 512, 2511, 64, 4), (96, 1536, 1188, 64, 2), (2, 32, 576, 64, 1), (64, 1024, 384, 128, 1), (48, 384, 733, 64, 1),
    # ... and of few rows they do not
    (8, 8, 1730, 128, 28), (8, 8, 2048, 128, 32), (8, 32, 8208, 128, 29), (2, 2, 640, 128, 10)])
def test_the_rows_of_a_step_weigh_in_its_splits(units, rows, Sk, D, splits):
    assert lowering._split_lengths(lowering.decode_even_split(units, Sk, D, rows=rows), Sk)[0] == splits


def test_few_counts_find_the_cheapest():
    """A call at a length not seen before evaluates at most ten counts, and the cheapest of all 64 is at most 4 % cheaper (0.2 %
    in the mean)."""
    excess = []
    for units in (1, 2, 8, 12, 32, 48, 64, 96, 128, 200, 256, 257, 512, 1040):
        for Sk in (1, 47, 95, 96, 200, 576, 1037, 2048, 5003, 16384, 65537):
            for rows, weight in ((1, 0.5), (1, 1.0), (4, 1.0), (16, 0.5), (16, 1.0)):
                counts = lowering._even_counts(units, Sk, weight, rows * units / 256)
                costs = [lowering._even_cost(n, units, Sk, weight, rows * units / 256) for n in range(1, max(1, min(64, Sk // 48)) + 1)]
                assert len(counts) <= 10 and min(counts) >= 1 and max(counts) <= len(costs)
                excess.append(min(costs[n - 1] for n in counts) / min(costs) - 1)
    assert max(excess) <= 0.04 and sum(excess) / len(excess) <= 0.002


def test_a_growing_cache_evaluates_its_splits_once_in_32_steps():
    lowering._even_best.cache_clear()
    for Sk in range(1, 1025):
        n = lowering.decode_even_split(8, Sk, 128, rows=32)
        splits, size = lowering._split_lengths(n, Sk)
        assert splits == 1 or size >= 64
    assert lowering._even_best.cache_info().misses <= 1024 // 32 + 1


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("splits", [2, 4, 5, 8, 9, 17, 33, 37, 64, 70])
def test_merge_of_any_number_of_splits(splits, D):
    """Fewer splits than a block's groups of threads take at a time, as many, a second round of some of the groups (from 33 splits at
    head dimension 128, 65 at 64), and a last group that has none; against float64 with the error of the unsplit step (fp32 sums: the order of the merge does not show in bf16),
    also where whole splits hold nothing but keys of probability 0 (a bias of -inf) and where a row sees a single key."""
    B, Hq, Hkv, S = 2, 6, 2, 64 * splits - 16
    g = torch.Generator(device="cuda").manual_seed(splits)
    q, k, v = (torch.randn(s, generator=g, device="cuda").bfloat16() for s in ((B, Hq, 1, D), (B, Hkv, S, D), (B, Hkv, S, D)))
    plan = AttnPlan(scale=D ** -0.5)
    kk, vv = (t.double().repeat_interleave(Hq // Hkv, 1) for t in (k, v))
    scores = torch.matmul(q.double(), kk.transpose(-1, -2).contiguous()) * plan.scale
    for live in (slice(0, S), slice(S // 2 + 5, S // 2 + 6), slice(S - 70, S - 3)):
        bias = torch.full((B, 1, 1, S), float("-inf"), device="cuda", dtype=torch.bfloat16)
        bias[..., live] = 0
        kw = {} if live == slice(0, S) else {"score_bias": bias}
        out = attention(q, k, v, plan, num_splits=splits, **kw)
        assert lowering.attention.last_launch["kernels"] == ["lf_attn_decode", "lf_attn_decode_combine"]
        assert lowering.attention.last_launch["grid"][1] == splits
        want = torch.matmul(torch.softmax(scores + bias.double(), dim=-1), vv)
        whole = attention(q, k, v, plan, num_splits=1, **kw)
        err, err_whole = ((x.double() - want).norm() / want.norm() for x in (out, whole))
        assert err <= 1.5 * err_whole + 2.0 ** -9       # either rounds once to bf16 and P to bf16 on the way


@pytest.mark.parametrize("B,Hkv,D,Sk,group,page,beats", [
    (2, 16, 64, 8930, 1, 1, True), (9, 24, 64, 5120, 1, 16, True), (60, 32, 128, 64, 1, 8, True),      # measured on both sides
    (64, 8, 128, 2048, 4, 16, True), (64, 4, 128, 2048, 8, 1, True),
    (66, 32, 128, 611, 2, 1, False), (281, 8, 128, 305, 4, 1, False), (269, 8, 128, 5602, 2, 1, False), (272, 8, 64, 129, 2, 1, True),
    (285, 4, 128, 144, 8, 1, True), (264, 8, 128, 496, 4, 16, False), (1, 8, 128, 8208, 4, 16, False), (1, 16, 128, 108, 1, 1, False)])
def test_cooperative_decode_is_chosen_where_it_is_faster(B, Hkv, D, Sk, group, page, beats):
    waves = 8 if Hkv % 8 == 0 else 4
    assert lowering.decode_coop_beats(B * Hkv // waves, waves, B * Hkv, Sk, group, page, D) == beats


@pytest.mark.gpu
@pytest.mark.parametrize("B,Hkv,D,Sk,group,page", [(2, 16, 64, 8931, 1, 1), (9, 24, 64, 2064, 2, 16), (60, 32, 128, 64, 1, 8),
                                                   (1, 8, 128, 20000, 1, 4), (3, 32, 128, 33, 3, 1)])
def test_steps_at_the_edges_of_the_rule(B, Hkv, D, Sk, group, page):
    """Few workgroups in many splits, a sequence of a few steps: both forms against float64 (P and the result are rounded to
    bf16, 2^-9 each), the rule's choice the bits of the form that it names."""
    n = Sk // page
    g = torch.Generator(device="cuda").manual_seed(Sk)
    q = torch.randn((B, Hkv * group, 1, D), generator=g, device="cuda").bfloat16()
    pool = (B * n, Hkv, D) if page == 1 else (B * n, page, Hkv, D)
    k, v = (torch.randn(pool, generator=g, device="cuda").bfloat16() for _ in range(2))
    table = torch.randperm(B * n, generator=g, device="cuda").view(B, n).to(torch.int32)
    kk, vv = (x[table.long()].reshape(B, n * page, Hkv, D).transpose(1, 2).double().repeat_interleave(group, 1) for x in (k, v))
    plan = AttnPlan(scale=D ** -0.5, k_paged=True, v_paged=True)
    want = torch.matmul(torch.softmax(torch.matmul(q.double(), kk.transpose(-1, -2).contiguous()) * plan.scale, dim=-1), vv)
    got = attention(q, k, v, plan, table, table)
    coop = bool(lowering.attention.last_launch["cooperative_loads"])
    assert coop == lowering.decode_coop_beats(B * Hkv // 8, 8, B * Hkv, Sk, group, page, D)
    for form in (True, False):
        out = attention(q, k, v, plan, table, table, choice={"head_per_wave": form})
        assert (out.double() - want).norm() / want.norm() <= 2.0 ** -8
        if form == coop:
            assert torch.equal(out, got)
