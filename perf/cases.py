"""Workloads the framework's speed is measured on, through its public entry points.

Five kinds of work, each over the range of sizes it is used at:

* ``prefill`` -- attention over whole prompts, written as the README of the user surface writes it and run through
  ``torch.compile(backend=loopfuse_backend)``: causal, causal sliding window or no mask, optional logit softcap,
  grouped query heads, bf16 / fp16, head dims 64 and 128, any sequence length.
* ``masked``  -- the same with the mask as a boolean tensor (a causal mask and the key padding of a batch of prompts
  of different lengths), the call ``F.scaled_dot_product_attention(q, k, v, attn_mask=...)``.
* ``train``   -- forward and backward of the attention of a training step, traced with gradients enabled.
* ``decode``  -- one new token per sequence against a KV cache, the direct operator of a serving loop
  (``lowering.attention``): contiguous caches and page pools of 1, 16 and 64 tokens per page.
* ``mlp``     -- the two linear layers around an attention, ``linear -> gelu -> linear``, which a graph without an
  attention runs on the generated kernels.

The backend runs with ``mode=None``, its fixed heuristics: the default mode times kernel variants on the first call
of a shape and may keep another one in another process.
"""
from __future__ import annotations

import functools
import math

import torch
import torch.nn.functional as F

from loopfuse_amd import loopfuse_backend
from loopfuse_amd.lowering import AttnPlan, attention

# every (shape class, options) pair below is a specialisation of its own of one traced function
torch._dynamo.config.recompile_limit = 256
torch._dynamo.config.accumulated_recompile_limit = 4096

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
_backend = functools.partial(loopfuse_backend, mode=None)


def _attn(kind, name, B, Hq, Hkv, S, D, dtype, mask="causal", window=0, softcap=0.0, page=0):
    c = {"kind": kind, "B": B, "Hq": Hq, "Hkv": Hkv, "S": S, "D": D, "dtype": dtype}
    if kind in ("prefill", "train"):
        c.update(mask=mask, window=window, softcap=softcap)
    if kind == "decode":
        c["page"] = page
    return {"name": name, **c} if name else c


def _mlp(name, M, width, hidden, dtype):
    c = {"kind": "mlp", "M": M, "width": width, "hidden": hidden, "dtype": dtype}
    return {"name": name, **c} if name else c


def listed():
    return [
        # a short batch (configuration 1's shape in bf16): launches and host work are what a user waits for
        _attn("prefill", "prefill_small", 2, 8, 8, 512, 64, "bf16"),
        # the headline configuration: a batch of 2k-token prompts, all heads with K/V of their own
        _attn("prefill", "prefill_causal", 8, 32, 32, 2048, 128, "bf16"),
        # the layers of models with local attention: window 256, grouped heads, softcap 30
        _attn("prefill", "prefill_window_cap", 8, 32, 8, 2048, 128, "bf16", mask="sliding", window=256, softcap=30.0),
        # one long prompt of a length nothing divides, grouped heads, fp16
        _attn("prefill", "prefill_long_ragged", 1, 32, 8, 6001, 128, "fp16"),
        # prompts of different lengths padded to one batch, the mask given as a tensor
        _attn("masked", "prefill_padded_mask", 4, 32, 32, 1536, 128, "bf16"),
        # the attention of a training step at the headline shape (half its batch)
        _attn("train", "train_causal", 4, 32, 32, 2048, 128, "bf16"),
        # a smaller model: head dim 64, grouped heads, a length that is no multiple of a tile
        _attn("train", "train_gqa_d64", 8, 16, 4, 1000, 64, "fp16"),
        # decode over a contiguous cache, every query head with K/V of its own
        _attn("decode", "decode_dense", 64, 32, 32, 2048, 128, "bf16"),
        # decode over a page pool, pages of 16 tokens, grouped heads
        _attn("decode", "decode_paged16", 64, 32, 8, 2048, 128, "bf16", page=16),
        # the reference's own paged format, one token per page, at its benchmark's grouping 32 / 4
        _attn("decode", "decode_paged1", 64, 32, 4, 2048, 128, "bf16", page=1),
        # one user's long conversation: a single sequence, latency counts
        _attn("decode", "decode_single", 1, 32, 8, 8208, 128, "bf16", page=16),
        # the tokens of one continuous-batching step through a 4096-wide block
        _mlp("mlp_step", 256, 4096, 16384, "bf16"),
    ]


def _pairs(case):
    """(query, key) pairs that are kept, for one head, summed over the batch."""
    B, S = case["B"], case["S"]
    if case["kind"] == "decode":
        return B * S
    if case["kind"] == "masked":
        return sum(n * (n + 1) // 2 + (S - n) * n for n in _lengths(case))
    if case["mask"] == "none":
        return B * S * S
    w = min(case["window"], S) if case["mask"] == "sliding" else S
    return B * (w * (w + 1) // 2 + (S - w) * w)


def _lengths(case):
    """Prompt lengths of a padded batch: spread over the upper half of S."""
    B, S = case["B"], case["S"]
    return [S - (S // 2) * b // max(B, 2) for b in range(B)]


def work(case):
    if case["kind"] == "mlp":
        M, w, h = case["M"], case["width"], case["hidden"]
        return {"bytes": 2 * (2 * M * w + 2 * w * h + w + h), "flops": 4 * M * w * h}
    B, Hq, Hkv, S, D = (case[k] for k in ("B", "Hq", "Hkv", "S", "D"))
    product = 2 * _pairs(case) * Hq * D
    q, kv = 2 * B * Hq * S * D, 2 * B * Hkv * S * D
    if case["kind"] == "decode":
        pages = 8 * B * (S // case["page"]) if case["page"] else 0      # two int32 tables
        return {"bytes": 2 * kv + 4 * B * Hq * D + pages, "flops": 2 * product}
    if case["kind"] == "train":      # two products forward, five backward; Q, dO, K, V in, O, dQ, dK, dV out
        return {"bytes": 4 * q + 4 * kv, "flops": 7 * product}
    mask = B * S * S if case["kind"] == "masked" else 0
    return {"bytes": 2 * q + 2 * kv + mask, "flops": 2 * product}


def _cost(case):
    w = work(case)
    return max(w["bytes"] / 5e12, w["flops"] / 6e14)


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    most = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(("prefill", "prefill", "masked", "train", "decode", "decode", "mlp"))
        dtype = rng.choice(("bf16", "bf16", "fp16"))
        if kind == "mlp":
            case = _mlp("", log(16, 8192), 64 * log(16, 128), 64 * log(32, 256), dtype)
        else:
            group = rng.choice((1, 1, 2, 4, 8))
            Hkv = rng.choice((2, 4, 8, 16, 32))
            D = rng.choice((64, 128, 128))
            if kind == "decode":
                page = rng.choice((0, 1, 16, 16, 64))
                S = log(256, 32768)
                S -= S % max(page, 1)
                case = _attn(kind, "", log(1, 128), Hkv * group, Hkv, max(S, 64), D, dtype, page=page)
            else:
                mask = rng.choice(("causal", "causal", "sliding", "none"))
                window = log(64, 1024) if mask == "sliding" else 0
                cap = rng.choice((0.0, 0.0, 30.0)) if kind == "prefill" else 0.0
                case = _attn(kind, "", log(1, 16), Hkv * group, Hkv, log(128, 8192), D, dtype, mask, window, cap)
            if Hkv * group > 64:
                continue
        if _cost(case) <= most:
            return case


# ---- the user's programs ---------------------------------------------------------------------------------

@functools.lru_cache(maxsize=None)
def _attention_program(mask, window, cap, groups, dynamic):
    def attn(q, k, v):
        if groups > 1:
            k = k.repeat_interleave(groups, dim=1)
            v = v.repeat_interleave(groups, dim=1)
        s = q @ k.transpose(-2, -1) * (q.shape[-1] ** -0.5)
        if cap:
            s = torch.tanh(s / cap) * cap
        if mask == "causal":
            s = torch.ops.loopfuse.causal_mask(s)
        elif mask == "sliding":
            s = torch.ops.loopfuse.sliding_mask(s, window)
        return torch.softmax(s, dim=-1) @ v

    return torch.compile(attn, backend=_backend, dynamic=dynamic)


@functools.lru_cache(maxsize=None)
def _masked_program(grouped):
    def attn(q, k, v, mask):
        return F.scaled_dot_product_attention(q, k, v, attn_mask=mask, enable_gqa=grouped)

    return torch.compile(attn, backend=_backend, dynamic=True)


@functools.lru_cache(maxsize=None)
def _mlp_program():
    def mlp(x, w1, b1, w2, b2):
        return F.linear(F.gelu(F.linear(x, w1, b1)), w2, b2)

    return torch.compile(mlp, backend=_backend, dynamic=True)


def prepare(case, seed):
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    dtype = _DTYPES[case["dtype"]]

    def normal(*shape, std=1.0):
        return torch.empty(shape, dtype=dtype, device=dev).normal_(0.0, std, generator=gen)

    if case["kind"] == "mlp":
        M, w, h = case["M"], case["width"], case["hidden"]
        return {"kind": "mlp", "fn": _mlp_program(),
                "args": (normal(M, w), normal(h, w, std=w ** -0.5), normal(h), normal(w, h, std=h ** -0.5), normal(w))}

    B, Hq, Hkv, S, D = (case[k] for k in ("B", "Hq", "Hkv", "S", "D"))
    if case["kind"] == "decode":
        page = case["page"]
        plan = AttnPlan(scale=D ** -0.5, k_paged=page > 0, v_paged=page > 0)
        q = normal(B, Hq, 1, D)
        if not page:
            return {"kind": "decode", "plan": plan, "args": (q, normal(B, Hkv, S, D), normal(B, Hkv, S, D)), "tables": ()}
        n = S // page
        pool = (B * n, Hkv, D) if page == 1 else (B * n, page, Hkv, D)
        table = torch.randperm(B * n, generator=gen, device=dev).view(B, n).to(torch.int32)
        return {"kind": "decode", "plan": plan, "args": (q, normal(*pool), normal(*pool)), "tables": (table, table.clone())}

    q, k, v = normal(B, Hq, S, D), normal(B, Hkv, S, D), normal(B, Hkv, S, D)
    group = Hq // Hkv
    if case["kind"] == "masked":
        order = torch.randperm(B, generator=gen, device=dev)
        lengths = torch.tensor(_lengths(case), device=dev)[order]
        pos = torch.arange(S, device=dev)
        mask = (pos[None, :] <= pos[:, None])[None, None] & (pos[None, :] < lengths[:, None])[:, None, None, :]
        return {"kind": "masked", "fn": _masked_program(group > 1), "args": (q, k, v, mask)}
    # a serving program sees every prompt length (dynamic shapes), a training step is traced for its own
    train = case["kind"] == "train"
    fn = _attention_program(case["mask"], case["window"], case["softcap"], group, not train)
    state = {"kind": case["kind"], "fn": fn, "args": (q, k, v)}
    if train:
        for t in (q, k, v):
            t.requires_grad_(True)
        state["dout"] = normal(B, Hq, S, D)
    return state


def run(state):
    kind = state["kind"]
    if kind == "train":
        out = state["fn"](*state["args"])
        return (out, *torch.autograd.grad(out, state["args"], state["dout"]))
    with torch.no_grad():
        if kind == "decode":
            q, k, v = state["args"]
            return attention(q, k, v, state["plan"], *state["tables"])
        return state["fn"](*state["args"])


def tolerance(case):
    # Inputs, probabilities and results are bf16 / fp16, every sum is fp32.  Measured against the same path in 64 bits:
    # bf16 2.4e-3 (gradients up to 6.3e-3 where the captured graph rounds every intermediate), fp16 6.1e-4 at most.
    if case["dtype"] == "fp16":
        return {"rel": 2.5e-3}
    return {"rel": 2.5e-2 if case["kind"] == "train" else 1e-2}
