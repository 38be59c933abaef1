"""Work splits of decode steps: ``lowering.decode_even_split`` and the merge with one block per output row."""
import pytest
import torch

from loopfuse_amd import lowering
from loopfuse_amd.lowering import AttnPlan, attention


def test_even_splits_stay_within_their_limits():
    """Splits of 48 keys at least and 64 of them at most; the sequence is covered; a short sequence and a launch that fills the
    CUs by itself are left whole; a long one of few units is split over all CUs."""
    for D in (64, 128):
        for units in (1, 2, 8, 24, 96, 255, 256, 257, 700):
            for Sk in (16, 47, 96, 208, 1000, 8208, 65536):
                n = lowering.decode_even_split(units, Sk, D)
                splits, size = lowering._split_lengths(n, Sk)
                assert 1 <= n <= 64 and (n == 1 or Sk // n >= 48) and splits * size >= Sk > (splits - 1) * size
        assert lowering.decode_even_split(256, 4000, D) == 1 and lowering.decode_even_split(4, 90, D) == 1
        assert lowering._split_lengths(lowering.decode_even_split(8, 20000, D), 20000)[0] >= 29
    for rows, nsplit in ((1, 1), (7, 4), (8, 5), (4097, 64)):
        for D in (64, 128):
            grid = lowering.decode_combine_grid(rows, nsplit, D)
            assert grid == rows or grid * (1024 // D) >= rows


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("splits", [2, 4, 5, 8, 9, 17, 33, 64])
def test_merge_of_any_number_of_splits(splits, D):
    """Fewer splits than a block's groups of threads take at a time, as many, more than one round of them, and a last group that
    has none; against float64 with the error of the unsplit step (fp32 sums: the order of the merge does not show in bf16),
    also where whole splits hold nothing but keys of probability 0 (a bias of -inf) and where a row sees a single key."""
    B, Hq, Hkv, S = 2, 6, 2, 64 * 64
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
        want = torch.matmul(torch.softmax(scores + bias.double(), dim=-1), vv)
        whole = attention(q, k, v, plan, num_splits=1, **kw)
        err, err_whole = ((x.double() - want).norm() / want.norm() for x in (out, whole))
        assert err <= 1.5 * err_whole + 2.0 ** -9       # either rounds once to bf16 and P to bf16 on the way
