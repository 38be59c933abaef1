"""Lowering: attention plan -> specialised gfx950 HIP kernel -> launcher.

This module is the counterpart of the reference's Triton emitter
(``loopfuse/codegen.py:100-126`` ``codegen_program`` and the generated
``launch_kernel_0``, ``codegen.py:215-298``).  Instead of printing a kernel per
graph it selects hand-written building blocks from ``csrc/kernels`` and
specialises them with ``-D`` options (dtype, head dim, mask kind, softcap,
paging, rows per unit); hipRTC compiles the result once per specialisation and
the code object is cached on disk.

Everything dynamic (batch, heads, sequence lengths, strides, scale, window,
softcap value) is a run-time kernel parameter, so a new sequence length does not
recompile (the reference makes every dimension a ``tl.constexpr``,
``codegen.py:394-396``).
"""
from __future__ import annotations

import ctypes
import dataclasses
import functools
import json
import math
import os
import threading
from typing import Optional

import torch

from . import runtime
from .skip import TILE_SHAPES

MASK_NONE, MASK_CAUSAL, MASK_SLIDING = 0, 1, 2
MASK_BITS = 8        # KernelSpec.bias of a call whose boolean mask the kernel reads as bits (lf_mask_bits.hip)
DECODE_QROWS = 16    # query rows one decode unit holds (the MFMA N dimension)
_MASK_NAMES = {"none": MASK_NONE, None: MASK_NONE, "causal": MASK_CAUSAL, "sliding": MASK_SLIDING}
_DTYPE_CODE = {torch.bfloat16: 0, torch.float16: 1}

# hipcc/hipRTC flags common to every kernel.  Packed-FP32 instruction selection
# (v_pk_*_f32) is switched off on purpose: scalar fp32 VALU code only.
COMMON_OPTS = ("-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops")


_ENVIRON = os.environ
_VARIABLES = _ENVIRON._data if os.name == "posix" and isinstance(getattr(_ENVIRON, "_data", None), dict) else None


def _env(name: str, default=None):
    """``os.environ.get``, without the exception that raises and catches for each variable that is not set: 0.6 us, half a
    dozen times per call of ``attention``.  (CPython's environment keeps its variables as bytes in ``_data``; another mapping
    put in its place is asked in the ordinary way.)"""
    if os.environ is _ENVIRON and _VARIABLES is not None and name.encode() not in _VARIABLES:
        return default
    return os.environ.get(name, default)


class AttnParams(ctypes.Structure):
    """Mirror of ``struct LfAttnParams`` in csrc/kernels/lf_common.hip.h."""

    _fields_ = (
        [(n, ctypes.c_void_p) for n in ("q", "k", "v", "o", "k_table", "v_table", "part_acc", "part_ml", "visits", "bias", "obias",
                                        "q2", "k2")]
        + [(n, ctypes.c_longlong) for n in (
            "q_sb", "q_sh", "q_ss", "k_sb", "k_sh", "k_ss", "v_sb", "v_sh", "v_ss", "o_sb", "o_sh", "o_ss",
            "bias_sb", "bias_sh", "bias_sq", "ob_sb", "ob_sh", "ob_sq",
            "q2_sb", "q2_sh", "q2_ss", "k2_sb", "k2_sh", "k2_ss", "k_span", "v_span")]
        + [(n, ctypes.c_int) for n in (
            "B", "Hq", "Hkv", "Sq", "Sk", "window", "kt_stride", "vt_stride", "nsplit", "rows", "split_len", "k2_group")]
        + [("scale", ctypes.c_float), ("softcap", ctypes.c_float), ("denom_add", ctypes.c_float)]
    )


@dataclasses.dataclass(frozen=True)
class KernelSpec:
    """Compile-time specialisation of one kernel family (= one code object)."""

    family: str            # "prefill" | "prefill_swp" | "decode" | "bwd"
    dtype: int             # 0 bf16, 1 fp16
    head_dim: int          # 64 | 128
    mask: int = MASK_NONE
    softcap: bool = False
    paged: int = 0         # bit 0: K paged, bit 1: V paged
    page_size: int = 1
    table_i64: bool = False
    rows: int = 1          # decode: query rows a unit can hold (fixed, the MFMA N dimension)
    waves: int = 4         # decode: waves per workgroup
    v_tr: bool = True      # prefill: transposed LDS reads for V
    headwave: bool = False  # decode: one kv head per wave (8 waves) instead of 4 waves sharing a head
    coop: bool = False     # decode, headwave: the workgroup loads whole 16-token blocks, rows reach the waves through LDS
    rowload: bool = False  # decode, register-staged path: whole-row non-temporal loads, K through a wave-private LDS tile
    denom: bool = False    # prefill: softmax denominator sum + c (c a run-time parameter)
    bias: int = 0          # prefill: bit 0 additive score bias tensor, bit 1 additive output bias tensor, bit 2 unaligned rows;
                           # prefill_swp: MASK_BITS a boolean mask as bits instead
    pack: int = 0          # prefill_swp, grouped-query attention: a workgroup's waves take 2 or 4 heads of one group
    page_size_v: int = 0   # tokens per page of the V pool when it differs from K's (0 = same)
    d2: int = 0            # prefill: depth of a second score product Q2 K2^T (0, 16, 32, 64)
    safe: bool = False     # rows that saw no key come out as zeros instead of NaN
    bn: int = 0            # prefill_swp: keys per LDS tile, 32 (three workgroups per CU) or 0 / 64 (two)
    extra: tuple = ()      # further -D options (tuning experiments)
    stay: bool = False     # prefill_swp, bwd: results by plain stores (prefill_out_stays, bwd_grads_stay)

    def __hash__(self):    # formed once: a call looks its kernels up by it, several times
        h = self.__dict__.get("_hash")
        if h is None:
            h = hash(tuple(getattr(self, f) for f in self.__dataclass_fields__))
            object.__setattr__(self, "_hash", h)
        return h

    def __getstate__(self):    # (strings hash otherwise in another process)
        return {k: v for k, v in self.__dict__.items() if k != "_hash"}

    def options(self) -> list[str]:
        o = list(COMMON_OPTS) + [
            f"-DLF_DTYPE={self.dtype}",
            f"-DLF_HEAD_DIM={self.head_dim}",
            f"-DLF_MASK={self.mask}",
            f"-DLF_SOFTCAP={int(self.softcap)}",
            f"-DLF_PAGED={self.paged}",
            f"-DLF_PAGE_SIZE={self.page_size}",
            f"-DLF_TABLE_I64={int(self.table_i64)}",
        ]
        if self.page_size_v:
            o += [f"-DLF_PAGE_SIZE_V={self.page_size_v}"]
        if self.family == "decode":
            o += [f"-DLF_DW={self.waves}", f"-DLF_HEADWAVE={int(self.headwave)}"]
            if self.coop:
                o += ["-DLF_COOP=1"]
            if self.rowload:
                o += ["-DLF_ROWLOAD=1"]
            if self.bias:
                o += ["-DLF_BIAS=1"]
        elif self.family == "prefill":
            o += [f"-DLF_V_TR={int(self.v_tr)}", f"-DLF_BIAS={self.bias}", f"-DLF_DENOM={int(self.denom)}"]
            if self.d2:
                o += [f"-DLF_D2={self.d2}"]
        elif self.family == "prefill_swp":
            if self.bn == 32:
                # 32-key tiles: 40 KB of LDS and <= 168 registers, so three workgroups share a CU
                o += ["-DLF_BN=32", "-DLF_WPE=3", "-DLF_KPF=3", "-DLF_VPF=2"]
            if self.pack:
                o += [f"-DLF_GQAPACK={int(self.pack)}"]
            if self.bias:
                o += ["-DLF_BIAS=2" if self.bias == MASK_BITS else "-DLF_BIAS=1"]
        if self.stay:
            o += ["-DLF_STAY=1"]
        if self.safe:
            o += ["-DLF_SAFE=1"]
        return o + list(self.extra)

    def files(self) -> tuple[str, ...]:
        kernel = {"prefill": "lf_attn_prefill.hip", "prefill_swp": "lf_attn_prefill_swp.hip",
                  "decode": "lf_attn_decode.hip", "bwd": "lf_attn_bwd.hip"}[self.family]
        if self.family == "decode":
            return ("lf_common.hip.h", kernel)
        # the two prefill kernels: their own tuning macros come first (the shared blocks use LF_BN)
        if self.family == "prefill_swp" and self.bias:
            # one code object holds the attention kernel and the kernel that reads the mask or the bias ahead of it
            return ("lf_common.hip.h", "lf_prefill_blocks.hip.h", kernel,
                    "lf_mask_bits.hip" if self.bias == MASK_BITS else "lf_bias_classify.hip")
        return ("lf_common.hip.h", "lf_prefill_blocks.hip.h", kernel)

    def entry(self) -> str:
        return {"prefill": "lf_attn_prefill", "prefill_swp": "lf_attn_prefill_swp", "decode": "lf_attn_decode",
                "bwd": "lf_attn_bwd_dq"}[self.family]

    def name(self) -> str:
        return (f"lf_{self.family}_t{self.dtype}_d{self.head_dim}_m{self.mask}_c{int(self.softcap)}"
                f"_p{self.paged}x{self.page_size}i{int(self.table_i64)}_r{self.rows}w{self.waves}v{int(self.v_tr)}h{int(self.headwave)}b{self.bias}n{int(self.denom)}"
                + (f"_q{self.d2}" if self.d2 else "") + (f"_gp{int(self.pack)}" if self.pack else "") + (f"_pv{self.page_size_v}" if self.page_size_v else "")
                + ("_z" if self.safe else "") + (f"_bn{self.bn}" if self.bn else "") + ("_co" if self.coop else "") + ("_rl" if self.rowload else "") + ("_st" if self.stay else "")
                + "".join("_" + e.replace("-D", "").replace("=", "") for e in self.extra))

    def source(self) -> str:
        return runtime.read_kernel_source(*self.files())


_spec = functools.lru_cache(maxsize=1024)(KernelSpec)      # (half the cost of making one)


@dataclasses.dataclass
class CompiledKernel:
    """What ``CODEGEN_ONLY`` returns in place of a runnable function (the
    reference returns ``KernelData(kernel_name, launch_name, code)``,
    ``loopfuse/codegen.py:66-71``)."""

    spec: KernelSpec
    code_object: bytes
    cache_hit: bool
    log: str

    @property
    def code(self) -> str:
        return "// options: " + " ".join(self.spec.options()) + "\n" + self.spec.source()


class CompiledKernels(list):
    """What a ``CODEGEN_ONLY`` call returns: the ``CompiledKernel`` of every fused call in
    the graph.  ``.code`` joins their sources, so the reference's usage
    ``print(compiled_fn(Q, K, V).code)`` (``tests/test_attention.py:28-29``) works as is."""

    @property
    def code(self) -> str:
        return "\n".join(k.code for k in self)


_compiled: dict[KernelSpec, CompiledKernel] = {}
_loaded: dict[tuple[KernelSpec, int], runtime.Module] = {}
_lock = threading.Lock()


def compile_spec(spec: KernelSpec, arch: str = runtime.DEFAULT_ARCH) -> CompiledKernel:
    """hipRTC-compile (or fetch from the on-disk cache) one specialisation.  Needs no GPU."""
    with _lock:
        ck = _compiled.get(spec)
    if ck is not None:
        return ck
    # outside the lock: different specialisations compile concurrently (the shim is re-entrant;
    # two threads asking for the same one both compile, the results are identical)
    code, hit, log = runtime.compile_source(spec.source(), spec.name(), spec.options(), arch)
    if spec.family == "bwd" and _env("USE_HARDCODE_KERNEL", "0") != "1":
        # the product kernels hand their accumulators to inline MFMAs as inputs: one that is spilled loses what the loop
        # added to it, and nothing at run time says so
        spilled = {name: n for name, n in runtime.private_segment_bytes(code).items() if n}
        if spilled:
            raise RuntimeError(f"loopfuse_amd: this compiler spills registers of the backward kernels ({spec.name()}: {spilled} "
                               "bytes per lane); their results would be wrong")
    ck = CompiledKernel(spec, code, hit, log)
    record = _env("LOOPFUSE_RECORD_SPECS")
    with _lock:
        if record and spec not in _compiled:
            # one JSON line per specialisation a workload asked for: specs_from_file() reads
            # them back, so a deployment can fill the code-object cache ahead of time
            with open(record, "a") as fh:
                fh.write(json.dumps(dataclasses.asdict(spec), sort_keys=True) + "\n")
        return _compiled.setdefault(spec, ck)


def specs_from_file(path: str) -> list[KernelSpec]:
    """Specialisations recorded with ``LOOPFUSE_RECORD_SPECS=<path>`` (duplicates dropped)."""
    seen: dict[KernelSpec, None] = {}
    with open(path) as fh:
        for line in fh:
            if line.strip():
                d = json.loads(line)
                d["extra"] = tuple(d.get("extra", ()))
                seen.setdefault(KernelSpec(**d))
    return list(seen)


def load_spec(spec: KernelSpec) -> runtime.Module:
    dev = torch.cuda.current_device()
    key = (spec, dev)
    mod = _loaded.get(key)
    if mod is None:
        ck = compile_spec(spec)
        with _lock:
            mod = _loaded.get(key)
            if mod is None:
                mod = runtime.Module(ck.code_object)
                _loaded[key] = mod
    return mod


_kernels: dict[tuple[KernelSpec, int], dict[str, runtime.Kernel]] = {}


def _kernels_of(spec: KernelSpec) -> dict:
    key = (spec, torch.cuda.current_device())
    named = _kernels.get(key)
    return _kernels.setdefault(key, {}) if named is None else named


def get_kernel(spec: KernelSpec, symbol: str, named: Optional[dict] = None) -> runtime.Kernel:
    """A kernel of a specialisation on the current device.  ``named``: ``_kernels_of(spec)``, for a caller that takes
    several (the key's hash costs 0.6 us)."""
    if named is None:
        named = _kernels_of(spec)
    k = named.get(symbol)
    if k is None:
        k = named[symbol] = load_spec(spec).kernel(symbol)
    return k


# ----------------------------------------------------------------------------
# plan
# ----------------------------------------------------------------------------

@dataclasses.dataclass
class AttnPlan:
    """What the front end extracts from a captured graph: the parameters of
    ``softmax(mask(mods(Q K^T))) V``.  ``scale`` multiplies the raw scores,
    ``softcap`` (if set) is applied as cap*tanh(s/cap) after scaling and before
    the mask, exactly the order of the reference graphs
    (``tests/benchmark.py:142-147``)."""

    mask: str | None = None            # None | "causal" | "sliding"
    window: int = 0
    scale: float = 1.0
    softcap: float | None = None
    k_paged: bool = False
    v_paged: bool = False
    denom_add: float = 0.0             # probabilities are e^(x-max) / (sum e^(x-max) + denom_add)
    zero_blind_rows: bool = False      # a row whose keys are all masked by the score bias gives zeros (as torch's
                                       # fused attention ops do) instead of the NaN of a softmax over -inf


class UnsupportedPlan(ValueError):
    """The shapes/dtypes cannot be served by the HIP kernels (caller falls back to eager)."""


def _check_tensor(name: str, t: torch.Tensor, dtype: torch.dtype) -> None:
    if not t.is_cuda:
        raise RuntimeError(f"loopfuse_amd: {name} is not on the GPU; the HIP path has no CPU fallback")
    if t.dtype != dtype:
        raise UnsupportedPlan(f"{name} has dtype {t.dtype}, expected {dtype}")
    if t.data_ptr() % 16:
        raise UnsupportedPlan(f"{name} is not 16-byte aligned")
    if t.is_contiguous() and t.shape[-1] % 8 == 0:
        return
    if t.stride(-1) != 1:
        raise UnsupportedPlan(f"{name} must have unit stride in its last dimension")
    for n, s in zip(t.shape[:-1], t.stride()[:-1]):
        if n > 1 and s % 8:
            raise UnsupportedPlan(f"{name} strides must be multiples of 8 elements (16-byte loads)")


_scratch: dict[tuple[int, int], torch.Tensor] = {}
_scratch_lock = threading.Lock()


def _get_scratch(device: torch.device, nfloats: int) -> torch.Tensor:
    """Split-K scratch, one buffer per (device, stream): launches on one stream are
    ordered, so they can share it (a step and its merge are launched under ``_scratch_lock``, or another
    thread's step on the stream could come between them); launches on different streams must not.  A graph keeps the address
    for all its replays, while the shared buffer is let go of when a later call needs a larger one, so a
    captured call takes its own from torch's allocator: what is allocated under capture stays the graph's."""
    if torch.cuda.is_current_stream_capturing():
        return torch.empty(nfloats, dtype=torch.float32, device=device)
    key = (device.index or 0, runtime.current_stream_handle())
    t = _scratch.get(key)
    if t is None or t.numel() < nfloats:
        t = torch.empty(max(nfloats, 1 << 20), dtype=torch.float32, device=device)
        _scratch[key] = t
    return t


def xcd_slots(units: int, tiles: int) -> int:
    """Grid of a kernel that maps its workgroups with ``lf_slot_of_block`` (csrc/kernels/lf_prefill_blocks.hip.h):
    8 XCDs x the slots of one, with the units cut into as many parts as that function chooses."""
    best = (units + 7) // 8 * tiles
    for t in (1, 2, 3):
        n = ((units << t) + 7) // 8 * ((tiles + (1 << t) - 1) >> t)
        if 17 * n <= 16 * best:
            best = n
    return 8 * best


def decode_split(units: int, Sk: int, cus: int = 256, per_cu: int = 2) -> int:
    """Number of KV splits across workgroups.  One workgroup per unit is enough once
    there are ``per_cu`` workgroups per CU (8 resident waves, each with 32 KB of loads
    in flight: two workgroups of 4 waves, or one of 8); below that the KV range is
    split, down to 512 tokens per split and up to 64 splits, and a second kernel merges
    the partial results."""
    env = _env("LOOPFUSE_DECODE_SPLITS")
    if env:
        return max(1, int(env))
    want = max(1, (per_cu * cus + units - 1) // units)
    if want > 4:
        # few units (small batch, long context): one workgroup per CU measured best
        want = max(4, (cus + units - 1) // units)
    most = max(1, min(64, Sk // 512))      # measured: >= 512 tokens per split, at most 64 splits
    return max(1, min(want, most))


def decode_even_split(units: int, Sk: int, D: int, cus: int = 256, rows: Optional[int] = None) -> int:
    """KV splits of a step whose four waves share a head (``units`` workgroups per split, ``rows`` output rows in all, one per
    unit unless given): the count with the least cost in a model, in keys of 128 streamed by a workgroup per CU, of
    - rounds of one workgroup per CU, each of a split's keys and 53 more at the head of it; a first round that is not full costs
      0.89 of one at least, a later one 0.78;
    - the merge launch, 235, and past four splits, where it takes one row per block, 44 and 34 per round of one row per CU;
    - the partials, 5.2 per split and round of one row per CU, and 0.9 per split past four.
    Up to one split per 48 keys, whose lengths are then rounded up to whole multiples of 32 (64 and more, the last what is left).
    Fitted on every count for 801 steps of 1 ... 512 units, 1 ... 64 rows each, 256 ... 30 000 keys, head dimensions 64 and 128: 0.9 %
    from the best measured count in the mean.  On 3446 other steps 0.870 of the time of splits of 512 keys, two workgroups per CU, in
    the mean, and slower than those by more than 3 % on 29 (12 % at worst); a model without the rows 0.883, 238 (25 %).  Splits of 512 keys /
    without rows / with them, us: D 64, 32 units of 16 rows 2511 keys 9.6 / 11.2 / 9.6, 96 of 16 1188 keys 10.2 / 12.8 / 10.1, 2 of 16 576
    keys 5.6 / 6.6 / 5.6; D 128, 8 units of 16 rows 2987 keys 13.2 / 9.9 / 9.3, of one row 1730 keys 12.1 / 7.2 / 7.2, of 4 rows 8208 keys
    13.4 / 12.3 / 12.3; 48 units of 16 rows, D 64, 25 814 keys 68.7 / 54.3 / 54.3."""
    # one evaluation for 32 lengths: a cache grows by a token per step, and a length that has not been seen costs 7 us
    return min(_even_best(units, (Sk + 31) // 32 * 32, D, units if rows is None else rows, cus), max(1, Sk // 48))


def _even_cost(n: int, units: int, Sk: int, weight: float, per_cu: float, cus: int = 256) -> float:
    size = (-(-Sk // n) + 31) // 32 * 32
    splits = -(-Sk // size)
    full, rest = divmod(units * splits, cus)
    t = (size + 53) * (full + (max(0.78 if full else 0.89, rest / cus) if rest else 0.0)) * weight
    if splits > 1:
        t += 235 + 5.2 * splits * per_cu * weight
        if splits > 4:
            t += 44 + 0.9 * splits + 34 * per_cu
    return t


def _even_counts(units: int, Sk: int, weight: float, per_cu: float, cus: int = 256) -> set:
    """The counts among which the cheapest is looked for: none, up to four splits (the merge's other form), those that fill one to
    four rounds of the CUs, the one at which a longer chain costs what the partials of another split do, and half of it.  All
    64 took 30 us of a call at a length not seen before, as each step of a growing cache has; these find a count within 0.2 % of the
    cheapest in the mean (4 % at worst), in 6."""
    most = max(1, min(64, Sk // 48))
    even = int(math.sqrt(0.89 * weight * Sk / (0.9 + 5.2 * per_cu * weight)))
    counts = (1, 2, 4, even, even // 2, cus // units, 2 * cus // units, 3 * cus // units, 4 * cus // units, most)
    return {max(1, min(most, n)) for n in counts} if most > 1 else {1}


@functools.lru_cache(maxsize=1024)
def _even_best(units: int, Sk: int, D: int, rows: int, cus: int = 256) -> int:
    weight, per_cu = D / 128, rows / cus
    return min([(_even_cost(n, units, Sk, weight, per_cu, cus), n) for n in _even_counts(units, Sk, weight, per_cu, cus)])[1]


def _even_time(units: int, Sk: int, D: int, rows: int, cus: int = 256) -> float:
    """Time of a step in the splits of ``decode_even_split`` as ``decode_coop_beats`` compares it, by the model that its
    constants were fitted to: CUs that stream a split's keys and 64 more at the head of it, a first round that is not full at
    nineteen twentieths, a later one at six tenths of a full one, the merge launch and its partials."""
    splits, size = _split_lengths(decode_even_split(units, Sk, D, cus, rows), Sk)
    full, rest = divmod(units * splits, cus)
    rounds = full + (max(0.6 if full else 0.95, rest / cus) if rest else 0.0)
    return (size + 64) * rounds * D / 128 + (230 if splits > 1 else 0) + (0.84 * splits if splits > 4 else 0)


def _coop_cost(n: int, units: int, Sk: int, rows: int, cus: int = 256) -> float:
    """Time of a decode step with cooperative loads in ``n`` KV splits (``units`` workgroups each), in tokens streamed by
    one workgroup per CU: rounds of one workgroup per CU, a last one that is not full costing nine tenths of one (fewer
    workgroups stream at their own rate, not at the card's), of a split's keys, the fill of its pipeline (160 tokens) and
    the partial results of its rows (8 each).  Constants fitted on 269 steps of 1 ... 128 sequences, 200 ... 16384 keys, 4 ... 32
    kv heads, pages of 1 ... 64 tokens: the count with the least cost is within 0.3 % of the best measured one in the mean (1.5 % at
    the 95th percentile) with token rows of 2 KB, within 1.6 % (10 %) with 1 KB."""
    splits, size = _split_lengths(n, Sk)
    full, rest = divmod(units * splits, cus)
    return (size + 160 + (8 * rows if n > 1 else 0)) * (full + (0.9 if rest else 0.0))


@functools.lru_cache(maxsize=1024)          # (every layer of a model asks for the same step)
def _coop_best(units: int, Sk: int, rows: int, cus: int = 256) -> tuple:
    """(splits, cost) of the cheapest count."""
    # one round of all CUs, of three quarters of them, two rounds, or no split; at least 160 tokens per split
    most = max(1, min(64, Sk // 160))
    cost, n = min((_coop_cost(n, units, Sk, rows, cus), n)
                  for n in {max(1, min(most, n)) for n in (1, cus // units, 3 * cus // (4 * units), 2 * cus // units)})
    return n, cost


def decode_coop_split(units: int, Sk: int, rows: int, cus: int = 256) -> int:
    """KV splits of a decode step with cooperative loads (``units`` workgroups per split)."""
    env = _env("LOOPFUSE_DECODE_SPLITS")
    if env:
        return max(1, int(env))
    return _coop_best(units, Sk, rows, cus)[0]


def decode_coop_fills(units: int, Sk: int, page_size: int) -> bool:
    most = min(8, Sk // 512) if page_size % 16 == 0 else min(32, Sk // 160)
    return units * max(1, most) >= 224


def decode_coop_pays(units: int, Sk: int, rows: int, page_size: int, cus: int = 256) -> bool:
    """Does a step with ``units`` workgroups per split pay with cooperative loads, against four waves per head in the splits of
    ``decode_split``, which steps in the library's static array and steps of a given number of splits make?
    First, there must be about as many workgroups as CUs.  Pages of 16 tokens and more, where the other form reads whole
    pages too: at up to 8 splits of 512 tokens (28 sequences of 4096 tokens, 8 heads, D 128: 79 against 84 us; 16 of 2048 32
    against 29).  Shorter pages: at up to 32 splits of 160 tokens (16 of 8192: 90 against 111 us).
    Second, the rounds must not be too empty nor the splits too short, against an even stream: less than 1.8 times with pages
    of 16 tokens and more, 2.4 times with shorter ones, which the other form reads in quarter rows.  Just over 256
    workgroups that cannot be split make a second round of a few (66 sequences of 228 tokens, 32 heads: 64 against 46 us; 92
    of 2192, 12 heads, pages of 16: 262 against 210), many short splits are mostly fill.  Of 454 steps, most of them next to
    the lines, 24 are more than 4 % slower than the other form without this, by up to 41 %, and 15 with it, by up to 12 %."""
    even = (1.8 if page_size % 16 == 0 else 2.4) * units * Sk
    return decode_coop_fills(units, Sk, page_size) and _coop_best(units, Sk, rows, cus)[1] * cus < even


def decode_coop_beats(units: int, waves: int, units_wave: int, Sk: int, rows: int, page_size: int, D: int) -> bool:
    """Is a step, its splits chosen by either form's own rule, faster with cooperative loads (``units`` workgroups of ``waves``
    heads per split) than with four waves per head (``units_wave`` workgroups)?  The costs of the two split rules, in tokens of
    one head, against each other, a token of the cooperative form at 0.6 of the other's time with pages of 16 tokens and more, at
    0.4 with shorter ones, which the other form reads in quarter rows.  Fitted on 470 steps and checked on 420 others of 64 ...
    32 768 keys: 0.46 and 0.42 % (short, long pages) off the faster form in the mean there, where ``decode_coop_pays`` was 2.4 %.
    Of the 107 steps that go the other way now, 0.90 of their time in the mean, three are 3 ... 4 % slower.  Before / now, us: 2
    sequences of 8930, 16 heads of 64, one-token pages 24.0 / 18.8; 9 of 5120, 24 heads of 64, pages of 16 60 / 48; 60 of 64, 32
    heads of 128, pages of 8 23.0 / 15.4.  A few workgroups more than CUs that are not split, pages shorter than 16: 8 heads of 128
    leave the second round to the other form, at any length (257 ... 287 workgroups, 305 ... 5602 keys: 1.04 ... 1.17 of its time; 264 of 611 keys
    156 against 137 us), half as many bytes per token do not (0.84 ... 1.04 from 128 keys on, 285 of 144 24.6 against 29.5).  Over 404 steps of
    257 ... 530 workgroups that is 0.6 % off the faster form in the mean there (by the costs 6.1, by ``decode_coop_pays`` 5.6); the costs
    are 0.5 % off with short pages from 288 workgroups on, with pages of 16 1.1 % up to there and 6 % beyond (7.6 by ``decode_coop_pays``).
    """
    if 256 < units < 288 and page_size % 16:
        return waves * D < 1024
    rate, fixed = (0.6, 50) if page_size % 16 == 0 else (0.4, 75)
    return rate * waves * D / 128 * _coop_best(units, Sk, rows)[1] + fixed < _even_time(units_wave, Sk, D, units_wave * rows)


def _split_lengths(n: int, Sk: int) -> tuple:
    """(splits, keys per split) of a decode step asked to make ``n``: whole pairs of 16-token steps."""
    size = (-(-Sk // n) + 31) // 32 * 32
    return -(-Sk // size), size


def decode_combine_grid(rows: int, nsplit: int, D: int) -> int:
    """Blocks of lf_attn_decode_combine: 256 threads, 4 consecutive d each; several rows to a block, or one row whose splits the
    block's groups of threads share, where there are more than they fetch at a time (4) and few rows."""
    per_block = 1024 // D
    return rows if nsplit > 4 and rows <= 4096 else -(-rows // per_block)


def static_split_runs(n: int, Sk: int, rows: int, D: int, room: int) -> bool:
    """Does a step asked to make ``n`` splits run with its partials in the library's static array of ``room`` bytes: it is
    split, and the partials (``rows`` output rows, D + 2 floats each per split) fit?"""
    upto = lambda region: (region + 255) // 256 * 256
    n = _split_lengths(n, Sk)[0]
    return n > 1 and upto(4 * rows * n * D) + upto(8 * rows * n) <= room


def decode_static_split(n: int, plain: int, Sk: int, rows: int, D: int, room: int) -> int:
    """KV splits of a step with cooperative loads whose partials live in the static array: ``n``, what
    ``decode_coop_split`` chose, where that runs; for an unsplit step ``plain``, what ``decode_split`` makes of it with
    the other loads; for one that does not fit the largest count that does.  So every step runs that one of the two rules
    can run there (``n`` is returned, to be refused, for one that no such count serves)."""
    runs = lambda m: static_split_runs(m, Sk, rows, D, room)
    if runs(n):
        return n
    if _split_lengths(n, Sk)[0] < 2:
        return plain if runs(plain) else n
    return next((m for m in range(n - 1, 1, -1) if runs(m)), n)


def _decode_headwave(paged: int, page_size: int, Hkv: int, D: int, P: "AttnParams", units_hw: int = 1 << 30,
                     Sk: int = 1 << 30, cus: int = 256) -> bool:
    """One kv head per wave pays when K and V are paged, token-major (head stride D,
    token stride Hkv*D), there are at least 8 heads to fill the 8 waves, and the
    (batch, head-chunk) units times at most 8 KV splits of >= 256 tokens still give one
    workgroup per CU (measured: below that, 4 waves per head with more splits win)."""
    env = _env("LOOPFUSE_DECODE_HEADWAVE")
    if env is not None:
        return env == "1"
    return (paged == 3 and Hkv % 8 == 0 and P.k_sh == D and P.v_sh == D
            and P.k_ss == Hkv * D and P.v_ss == Hkv * D
            and units_hw * max(1, min(8, Sk // 512)) >= cus)


def _decode_coop_waves(paged: int, page_size: int, page_size_v: int, bias_bits: int, Hkv: int, P: "AttnParams", D: int) -> int:
    """Waves of a workgroup that reads every 16-token block of its heads as one contiguous piece per token, one kv head
    per wave, and hands the rows to the waves through LDS (``-DLF_COOP=1``): 8, 4 (Hkv a multiple of 4 only), or 0 where
    that form does not serve the call -- pools of different page sizes, a score bias to carry along, heads of a token
    not side by side (a permuted [pages, Hkv, page, D] pool view goes to the per-wave loads, which follow the head
    stride), or less than 1 KB per token row, where a wave would need the page ids of several tokens per load (and
    where it gains nothing with longer pages: 4 heads of 64, 34 against 28 us).  A wave that fetches its own head reads 256-byte pieces 2 KB apart, which costs
    about a tenth of the HBM rate.  LOOPFUSE_DECODE_COOP=0 keeps the per-wave loads."""
    if paged != 3 or page_size_v or bias_bits or _env("LOOPFUSE_DECODE_COOP", "1") != "1":
        return 0
    if P.k_sh != D or P.v_sh != D or (page_size > 1 and (P.k_ss < Hkv * D or P.v_ss < Hkv * D)):
        return 0
    waves = 8 if Hkv % 8 == 0 else (4 if Hkv % 4 == 0 else 0)
    return 0 if waves * D < 512 else waves


def _decode_rowload(paged: int, page_size: int, page_size_v: int, bias_bits: int) -> bool:
    """The register-staged decode path reads whole rows (every 128-byte line in one piece) with
    non-temporal loads and passes K through a wave-private LDS tile (``-DLF_ROWLOAD=1``) when a
    16-token step lies inside one page (or K/V are dense) and there is no score bias.
    LOOPFUSE_DECODE_ROWLOAD=0 keeps the loads in MFMA operand layout."""
    if _env("LOOPFUSE_DECODE_ROWLOAD", "1") != "1" or bias_bits:
        return False
    return not paged or (page_size % 16 == 0 and (page_size_v or page_size) % 16 == 0)


def prefill_kv_tile(D: int, bias_bits: int = 0, choice: Optional[dict] = None, workgroups: int = 1 << 30,
                    keys: int = 1 << 30) -> int:
    """Keys per LDS tile of lf_attn_prefill_swp: 0 (the kernel's 64) or 32.  With 32-key tiles a
    workgroup needs 40 KB of LDS and at most 168 registers per lane, so three workgroups instead of
    two share a CU.  ``keys`` = most keys a query can see (the sequence or the window).  At head dimension 128 that pays
    once the launch has three workgroups for every CU (768): a third workgroup hides prologues and drains.  Long walks
    have few of these, and there two per CU and a shorter tail win until the launch has 2048 workgroups.  Times with 32
    over times with 64, geometric mean (extremes) over 320 launches with and without masks, caps and packed heads:
    768 ... 2047 workgroups, up to 700 keys 0.90 (0.80 ... 1.10), 700 ... 2047 0.97 (0.90 ... 1.04), 2048 and more 1.02 (0.94 ... 1.13: 784
    workgroups of 6211 keys; one 6001-token prompt, 1504 workgroups, 328 against 312 us); from 2048 workgroups on 0.95
    (0.79 ... 1.05); 500 ... 767 either way (0.72 ... 1.15).  At head
    dimension 64 it does not pay.  The bias tile classes of a score bias are per 64 keys, so biased calls keep 64.  So does a
    boolean mask, for its error: the exponents' first offset is the maximum of the first tile, and over 32 keys the largest weight
    is less often exactly 1 (relative 2-norm against float64, 64 / 32 keys: bf16 1024 keys 2.338e-3 / 2.346e-3, 300 keys with
    inputs of 6 1.821e-3 / 1.901e-3); a padding mask of 4 x 32 heads x 1536 takes 101 and 92 us, 110 before its bits.
    ``choice["bn"]`` (the tuner) or ``LOOPFUSE_BN`` override the default without a bias or mask."""
    if bias_bits:
        return 0
    want = (choice or {}).get("bn", _env("LOOPFUSE_BN"))
    if want is not None:
        return 32 if int(want) == 32 else 0
    return 32 if D == 128 and workgroups >= (3 * 256 if keys < 2048 else 8 * 256) else 0


def prefill_out_stays(nbytes: int) -> bool:
    """Does lf_attn_prefill_swp write an output of so many bytes by plain stores (``-DLF_STAY=1``), which leave it near whoever reads
    it next, and not in whole rows past the caches?  Whole over plain, the kernel with an element-wise kernel or a product
    behind it, over 40 launches: below 5 MB 0.98 ... 1.12, 5 ... 6 MB 0.96 ... 1.05, 6 ... 10 MB 0.91 ... 1.01, above 0.94 ... 1.03; the
    kernel alone 0.97 ... 1.03, 0.97 ... 1.00, 0.88 ... 1.00 and 0.91 ... 1.03."""
    return nbytes < 6_000_000


def prefill_variant(Sq: int, v_tr: bool = True) -> str:
    """Which prefill kernel serves a call.  Default: the software-pipelined kernel
    with direct-to-LDS staging (``prefill_swp``; dense K/V only, ``attention`` falls
    back to ``prefill`` for paged operands).  LOOPFUSE_PREFILL=w32 selects the
    register-staged kernel for comparison."""
    env = _env("LOOPFUSE_PREFILL", "swp")
    if not v_tr or env == "w32":
        return "prefill"
    return "prefill_swp"


# ---------------------------------------------------------------------------
# launch-heuristic tuning (the reference autotunes tile sizes with triton.autotune,
# loopfuse/codegen.py:355-404; the HIP kernels have fixed tiles, what varies here is
# which kernel variant and which work split serve a shape)
# ---------------------------------------------------------------------------
_tuned: dict = {}
_TUNE_FILE = os.path.join(runtime.CACHE_DIR, "autotune.json")


@functools.lru_cache(maxsize=None)
def _rules_version() -> str:
    """Digest of the kernels' sources and of the rules in this file: a choice measured before either changed was measured among
    other candidates, against another default, and is not taken from the file any more."""
    import hashlib
    h = hashlib.sha256()
    for path in [os.path.join(runtime.KERNEL_DIR, f) for f in sorted(os.listdir(runtime.KERNEL_DIR))] + [__file__]:
        if os.path.isfile(path):
            with open(path, "rb") as fh:
                h.update(fh.read())
    return h.hexdigest()[:12]


def _tune_key(q, k, plan: AttnPlan, k_table, bias_bits: int) -> str:
    B, Hq, Sq, D = q.shape
    if plan.k_paged:
        Hkv = k.shape[-2]
        Sk = k_table.shape[1] * (k.shape[1] if k.dim() == 4 else 1)
        ps = k.shape[1] if k.dim() == 4 else 1
    else:
        Hkv, Sk, ps = k.shape[1], k.shape[2], 0
    bucket = lambda n: 1 << max(0, (int(n) - 1)).bit_length()       # next power of two
    return (f"{q.dtype}|D{D}|m{plan.mask}|c{int(plan.softcap is not None)}|p{int(plan.k_paged)}{int(plan.v_paged)}x{ps}"
            f"|B{bucket(B * Hkv)}|g{Hq // Hkv}|q{bucket(Sq)}|k{bucket(Sk)}|b{bias_bits}|r{_rules_version()}")


def _load_tuned() -> None:
    if not _tuned and os.path.exists(_TUNE_FILE):
        try:
            import json
            with open(_TUNE_FILE) as fh:
                _tuned.update({key: choice for key, choice in json.load(fh).items() if key.endswith(f"|r{_rules_version()}")})
        except (OSError, ValueError, AttributeError):
            pass


def tuned_attention(q, k, v, plan: AttnPlan, k_table=None, v_table=None, **kw):
    """``attention`` with the launch heuristics chosen by measurement: on the first call
    of a shape class each candidate is timed on the call's own tensors (HIP events, a few
    launches), the winner is remembered in the process and, until a kernel or a rule changes, in
    ``autotune.json`` beside the code-object cache.  Used by the backend under ``mode="max-autotune"``."""
    if kw.get("score_bias") is not None or kw.get("score_mask") is not None or kw.get("out_bias") is not None or kw.get("record_visits") \
            or kw.get("force_family") or kw.get("num_splits") or kw.get("choice") or plan.denom_add != 0.0 or kw.get("q2") is not None:
        return attention(q, k, v, plan, k_table, v_table, **kw)
    _load_tuned()
    key = _tune_key(q, k, plan, k_table, 0)
    if key not in _tuned and q.is_cuda and torch.cuda.is_current_stream_capturing():
        # timing needs a host synchronisation, which a stream capture forbids: fixed heuristics
        return attention(q, k, v, plan, k_table, v_table, **kw)
    if key not in _tuned:
        B, Hq, Sq, D = q.shape
        Hkv = k.shape[-2] if plan.k_paged else k.shape[1]
        group = Hq // max(Hkv, 1)
        decode = plan.mask is None and ((Sq == 1 and group <= 64) or (group == 1 and Sq <= 16))
        if decode:
            cands = [{"head_per_wave": hw, "splits": sp} for hw in ((False, True) if plan.k_paged and plan.v_paged else (False,))
                     for sp in (None, 1, 2, 4, 8)]
        elif not (plan.k_paged or plan.v_paged):
            # kernel family, tile shape (keys per LDS tile, which also sets how many workgroups share a
            # CU; the reference's tuner searches tile sizes, codegen.py:360-393) and, for grouped query
            # heads, the packed / unpacked q tile
            cands = [{"prefill": "swp", "bn": 32}, {"prefill": "swp", "bn": 64}, {"prefill": "w32"}]
            if group % 2 == 0:
                cands[2:2] = [{"prefill": "swp", "bn": 32, "pack": False}, {"prefill": "swp", "bn": 64, "pack": False}]
        elif Sq > 1:
            cands = [{"bn": 32}, {"bn": 64}]
        else:
            cands = [{}]
        best, best_t = cands[0], float("inf")
        if len(cands) > 1:
            out = kw.get("out")
            for c in cands:
                c = {a: b for a, b in c.items() if b is not None}
                try:
                    for _ in range(2):
                        out = attention(q, k, v, plan, k_table, v_table, **{**kw, "out": out, "choice": c})
                    a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                    a.record()
                    for _ in range(5):
                        attention(q, k, v, plan, k_table, v_table, **{**kw, "out": out, "choice": c})
                    b.record()
                    b.synchronize()
                    t = a.elapsed_time(b)
                except UnsupportedPlan:
                    continue
                if t < best_t:
                    best, best_t = c, t
        _tuned[key] = best
        try:
            import json
            os.makedirs(os.path.dirname(_TUNE_FILE), exist_ok=True)
            with open(_TUNE_FILE, "w") as fh:
                json.dump(_tuned, fh, indent=0, sort_keys=True)
        except OSError:
            pass
    return attention(q, k, v, plan, k_table, v_table, **{**kw, "choice": _tuned[key]})


# ---------------------------------------------------------------------------
# launches kept per call signature
# ---------------------------------------------------------------------------
# What ``attention`` and ``attention_backward`` launch depends on shapes, strides, dtypes and alignment of their operands, the
# plan, the options of the call and the switches in the environment, on nothing else: a call whose signature was seen before
# repeats the launches recorded then, with its own pointers and new results.  Host time of a split decode step over a page pool
# 30 -> 16.5 us, of a small compiled prefill 67 -> 35 us (with the views and the plan of its graph formed once, AttentionMatch).
# Only calls that ran to their end are recorded, so what is refused is refused again; bounded, and emptied when full.
_SWITCHES = tuple(n.encode() for n in (
    "LOOPFUSE_BIAS_COPY", "LOOPFUSE_BIAS_TILES", "LOOPFUSE_BN", "LOOPFUSE_CHECK_TABLES", "LOOPFUSE_DECODE_COOP", "LOOPFUSE_DECODE_HEADWAVE",
    "LOOPFUSE_DECODE_ROWLOAD", "LOOPFUSE_DECODE_SPLITS", "LOOPFUSE_DECODE_WAVES", "LOOPFUSE_GQAPACK", "LOOPFUSE_KOPTS",
    "LOOPFUSE_PAGED_SWP", "LOOPFUSE_PREFILL", "LOOPFUSE_RECORD_SPECS", "USE_HARDCODE_KERNEL"))
_MAX_KEPT = 512
_NO_ROOM_CALLS = 1000      # calls of a backward that found no room for dS until it looks for it again
_kept: dict = {}
_PLAIN = (int, float, str, bool, type(None))
_PLAIN_TYPES = frozenset(_PLAIN)



def _signature(kind: str, tensors, plan: AttnPlan, options: Optional[dict]):
    """Key of a call over tensors on the GPU (None in the place of one that is not given); None: not to be kept."""
    if os.environ is not _ENVIRON or _VARIABLES is None:
        return None
    operands = []
    for t in tensors:
        if t is None:
            operands.append(None)
        elif not t.is_cuda or t.data_ptr() % 16:
            return None
        else:
            operands.append((t.shape, t.stride(), t.dtype, t.get_device()))
    fields = (plan.mask, plan.window, plan.scale, plan.softcap, plan.k_paged, plan.v_paged, plan.denom_add, plan.zero_blind_rows)
    choice = tuple(options.items()) if options else ()
    if not _PLAIN_TYPES.issuperset(map(type, fields)) and not all(isinstance(x, _PLAIN) for x in fields):
        return None
    for _, x in choice:
        if not isinstance(x, _PLAIN):
            return None
    return (kind, fields, choice, runtime.current_device(), tuple(map(_VARIABLES.get, _SWITCHES)), tuple(operands))


class _Kept:
    """The launches of one signature.  ``params``: the parameter block, its pointers still to be set; ``results``: shape and
    dtype of what a call allocates; ``scratch``: floats of split-K partials and where their second array starts; ``calls``: how
    often the record serves (None: as long as it is kept)."""

    __slots__ = ("params", "launches", "results", "scratch", "record", "calls")

    def __init__(self, params, steps, results, record, scratch=None, calls=None):
        self.params, self.launches, self.results = bytes(params), runtime.LaunchList(steps), results
        self.scratch, self.record, self.calls = scratch, record, calls

    def attention(self, q, k, v, k_table, v_table, out, lse):
        P = AttnParams.from_buffer_copy(self.params)
        if out is None:
            out = torch.empty(self.results[0], dtype=self.results[1], device=q.device)
        P.q, P.k, P.v, P.o = q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr()
        if k_table is not None:
            P.k_table = k_table.data_ptr()
        if v_table is not None:
            P.v_table = v_table.data_ptr()
        if self.scratch is not None:
            with _scratch_lock:        # no other thread's step on this stream between the launches
                scratch = _get_scratch(q.device, self.scratch[0])
                P.part_acc = scratch.data_ptr()
                P.part_ml = scratch.data_ptr() + self.scratch[1]
                self.launches.launch(P)
        else:
            P.part_ml = None if lse is None else lse.data_ptr()
            self.launches.launch(P)
        _last_launch.set(self.record)
        return out


def _keep(key, kept: _Kept) -> None:
    if len(_kept) >= _MAX_KEPT:
        _kept.clear()
    _kept[key] = kept


class _LastLaunch:
    """What the calling THREAD's last ``attention`` call launched (kernels, grid, block, tile
    shape): ``attention.last_launch["kernels"]``.  Each thread sees its own record."""

    def __init__(self):
        self._tls = threading.local()

    def set(self, record: dict) -> None:
        self._tls.record = record

    def _get(self) -> dict:
        return getattr(self._tls, "record", {})

    def __getitem__(self, key):
        return self._get()[key]

    def get(self, key, default=None):
        return self._get().get(key, default)

    def __repr__(self) -> str:
        return repr(self._get())


_last_launch = _LastLaunch()


def _on_device_of_first_argument(fn):
    """Kernel modules, the stream and the split-K scratch are looked up for the current
    device: make the device of Q current for the duration of the call when it is not."""
    @functools.wraps(fn)
    def guarded(q, *args, **kw):
        if isinstance(q, torch.Tensor) and q.is_cuda and q.get_device() != runtime.current_device():
            with torch.cuda.device(q.device):
                return fn(q, *args, **kw)
        return fn(q, *args, **kw)
    guarded.last_launch = _last_launch
    return guarded


@_on_device_of_first_argument
def attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, plan: AttnPlan,
              k_table: Optional[torch.Tensor] = None, v_table: Optional[torch.Tensor] = None,
              *, out: Optional[torch.Tensor] = None, record_visits: bool = False,
              force_family: str | None = None, num_splits: int | None = None, v_tr: bool = True,
              score_bias: Optional[torch.Tensor] = None, out_bias: Optional[torch.Tensor] = None,
              choice: Optional[dict] = None, merge_splits: bool = True,
              q2: Optional[torch.Tensor] = None, k2: Optional[torch.Tensor] = None,
              static_scratch: bool = False, lse: Optional[torch.Tensor] = None,
              score_mask: Optional[torch.Tensor] = None, mask_keep: bool = True):
    """Run fused attention on the GPU.

    q : [B, Hq, Sq, D];  k, v : [B, Hkv, Sk, D], or page pools [N, P, Hkv, D]
    ([N, Hkv, D] for one-token pages) with ``k_table``/``v_table`` [B, Sk/P].
    ``score_bias`` (broadcastable to [B, Hq, Sq, Sk], key stride 1) is added to the
    scaled / capped scores before the mask, ``out_bias`` (broadcastable to
    [B, Hq, Sq, D]) to the result -- the reference's "modified attention" graph
    (tests/test_accuracy.py:172-196).  Both are served by ``lf_attn_prefill`` only.
    ``score_mask`` (torch.bool, broadcastable to [B, Hq, Sq, Sk]; not together with ``score_bias``) stands for the score
    bias that is 0 where a key is visible -- True, or False with ``mask_keep=False`` -- and -inf elsewhere.
    ``q2`` [B, Hq, Sq, D2] and ``k2`` [B, H2, Sk, D2] (H2 divides Hq; D2 in 16, 32, 64) add a
    second product to the scores, ``Q K^T + Q2 K2^T`` before the scale -- the two-part scores
    of multi-head latent attention (reference tests/test_attention.py:126-151); served by
    ``lf_attn_prefill`` with dense K2.
    ``merge_splits=False`` leaves the partial results of a split decode unmerged (the
    output is then not written): for timing the streaming kernel alone.
    ``static_scratch=True`` (split decode only, ``out`` given): the step goes through the C ABI's
    ``lf_launch_decode_static``, whose split-K partials live in a static device array of the
    library -- no device memory is allocated anywhere in the call; a step whose partials exceed
    that array raises ``runtime.ShimError``.
    ``lse`` (float32 [B, Hq, Sq], contiguous): also write each row's log-sum-exp of the scaled,
    masked scores, in log2 units -- what ``attention_backward`` recomputes the probabilities
    from.  Served by ``lf_attn_prefill_swp`` (dense K/V); anything else raises ``UnsupportedPlan``.
    ``choice`` overrides the launch heuristics (what ``tuned_attention`` searches over):
    ``{"prefill": "swp" | "w32"}``, ``{"head_per_wave": bool, "splits": n}``.
    Returns O [B, Hq, Sq, D] and, with ``record_visits``, the uint8 record of the KV tiles
    each workgroup walked, ``[B * heads * q_tiles, kv_tiles]`` with ``heads = Hq`` and
    128-row q tiles, or ``heads = Hq / g`` and ``128 / g``-row q tiles when g = 2 or 4 query heads
    are packed (``last_launch["heads_per_workgroup"] == g``).
    """
    key = None
    if not (record_visits or static_scratch) and force_family is None and num_splits is None and v_tr and merge_splits \
            and score_bias is None and out_bias is None and q2 is None and k2 is None and score_mask is None:
        key = _signature("fwd", (q, k, v, k_table, v_table, out, lse), plan, choice)
        kept = _kept.get(key)
        if kept is not None:
            return kept.attention(q, k, v, k_table, v_table, out, lse)
    choice = choice or {}
    dtype = q.dtype
    if dtype not in _DTYPE_CODE:
        raise UnsupportedPlan(f"dtype {dtype} not supported by the MFMA kernels (bf16/fp16 only)")
    if q.dim() != 4:
        raise UnsupportedPlan("Q must be [B, Hq, Sq, D]")
    B, Hq, Sq, D = q.shape
    if D not in (64, 128):
        # Other head dimensions up to 128 (the reference takes any static D, ops.py:370-397): dense operands
        # are copied into zero-padded rows of 64 / 128 elements -- zeros add nothing to Q K^T, and the padded
        # columns of V give output columns that are cut off again -- at O(S D) beside the O(S^2 D) attention.
        Dp = 64 if D < 64 else 128
        if D > 128 or D < 1 or plan.k_paged or plan.v_paged or lse is not None or q2 is not None or static_scratch \
                or k.dim() != 4 or v.dim() != 4 or k.shape[-1] != D or v.shape[-1] != D:
            raise UnsupportedPlan(f"head dim {D} not supported (64 and 128; up to 128 by padding for dense operands)")
        grow = lambda t: None if t is None else torch.nn.functional.pad(t, (0, Dp - D))
        res = attention(grow(q), grow(k), grow(v), plan, None, None, record_visits=record_visits, score_bias=score_bias,
                        score_mask=score_mask, mask_keep=mask_keep, out_bias=grow(out_bias), force_family=force_family, num_splits=num_splits, v_tr=v_tr,
                        choice=choice, merge_splits=merge_splits)
        o_p, vis = res if record_visits else (res, None)
        if out is None:
            out = o_p[..., :D].contiguous()
        else:
            out.copy_(o_p[..., :D])
        return (out, vis) if record_visits else out
    if not (plan.scale > 0.0) or not math.isfinite(plan.scale):
        raise UnsupportedPlan("score scale must be positive and finite")
    softcap = None
    if plan.softcap is not None:
        # cap * tanh(s / cap) is even in cap: a negative cap (pre- and post-factor both negative
        # in the graph) is served as its magnitude; zero or a non-finite cap is not a softcap
        softcap = abs(float(plan.softcap))
        if not (softcap > 0.0) or not math.isfinite(softcap):
            raise UnsupportedPlan("softcap must be finite and non-zero")
    _check_tensor("Q", q, dtype)
    _check_tensor("K", k, dtype)
    _check_tensor("V", v, dtype)
    for name, t in (("K", k), ("V", v), ("K page table", k_table), ("V page table", v_table), ("score bias", score_bias),
                    ("score mask", score_mask), ("output bias", out_bias), ("Q2", q2), ("K2", k2), ("O", out)):
        if t is not None and t.device != q.device:
            raise RuntimeError(f"loopfuse_amd: {name} is on {t.device}, Q on {q.device}")

    P = AttnParams()
    paged = 0
    page_size = 1          # K pool (both pools when they agree)
    page_size_v = 0        # V pool, when it differs from K's
    table_i64 = False

    def kv_layout(t: torch.Tensor, table: Optional[torch.Tensor], is_paged: bool, which: str):
        nonlocal paged, page_size, page_size_v, table_i64
        if not is_paged:
            if t.dim() != 4 or t.shape[0] != B or t.shape[3] != D:
                raise UnsupportedPlan(f"{which} must be [B, Hkv, Sk, D]")
            return t.shape[1], t.shape[2], t.stride(0), t.stride(1), t.stride(2), None, 0
        if table is None or table.dim() != 2 or table.shape[0] != B:
            raise UnsupportedPlan(f"{which} page table must be [B, pages]")
        if table.dtype not in (torch.int32, torch.int64):
            raise UnsupportedPlan("page table must be int32 or int64")
        if not table.is_cuda:
            raise RuntimeError(f"loopfuse_amd: {which} page table is not on the GPU")
        if table.stride(1) != 1:
            table = table.contiguous()
        if _env("LOOPFUSE_CHECK_TABLES", "0") == "1" and table.numel():
            # debugging aid (waits for the stream): the kernels trust page ids, an id outside
            # the pool is a read outside the allocation
            lo, hi = int(table.min()), int(table.max())
            if lo < 0 or hi >= t.shape[0]:
                raise ValueError(f"loopfuse_amd: {which} page table holds ids in [{lo}, {hi}] for a pool of {t.shape[0]} pages")
        if t.dim() == 3:       # [N, Hkv, D], one token per page (the reference's format)
            ps, hk, sp, st, sh = 1, t.shape[1], t.stride(0), 0, t.stride(1)
        elif t.dim() == 4:     # [N, P, Hkv, D]
            ps, hk, sp, st, sh = t.shape[1], t.shape[2], t.stride(0), t.stride(1), t.stride(2)
        else:
            raise UnsupportedPlan(f"{which} pool must be [N, Hkv, D] or [N, P, Hkv, D]")
        if t.shape[-1] != D:
            raise UnsupportedPlan(f"{which} pool has head dim {t.shape[-1]}, Q has {D}")
        if ps & (ps - 1):
            raise UnsupportedPlan("page size must be a power of two")
        i64 = table.dtype == torch.int64
        if paged and table_i64 != i64:
            raise UnsupportedPlan("K and V page tables must share their dtype")
        if which == "V" and paged and ps != page_size:
            page_size_v = ps               # pools with different page sizes
        else:
            page_size = ps
        table_i64 = i64
        paged |= 1 if which == "K" else 2
        return hk, table.shape[1] * ps, sp, sh, st, table, table.stride(0)

    Hkv, Sk, P.k_sb, P.k_sh, P.k_ss, kt, P.kt_stride = kv_layout(k, k_table, plan.k_paged, "K")
    Hkv2, Sk2, P.v_sb, P.v_sh, P.v_ss, vt, P.vt_stride = kv_layout(v, v_table, plan.v_paged, "V")
    if Hkv != Hkv2 or Sk != Sk2:
        raise UnsupportedPlan("K and V disagree on heads or length")
    if Hq % Hkv:
        raise UnsupportedPlan("Hq must be a multiple of Hkv")
    group = Hq // Hkv
    mask = _MASK_NAMES[plan.mask]
    if mask == MASK_SLIDING and plan.window < 1:
        raise UnsupportedPlan("sliding mask needs window >= 1")

    if Sk < 1:
        # softmax over no keys is 0/0 in the eager graph: nothing a kernel should invent
        raise UnsupportedPlan("attention over an empty key sequence")
    if out is None:
        out = torch.empty((B, Hq, Sq, D), dtype=dtype, device=q.device)
    else:
        _check_tensor("O", out, dtype)
        if tuple(out.shape) != (B, Hq, Sq, D):
            raise UnsupportedPlan(f"O must be [{B}, {Hq}, {Sq}, {D}]")
    if B == 0 or Hq == 0 or Sq == 0:
        # no query rows: the (empty) output is the whole result, nothing to launch
        _last_launch.set({"kernels": [], "grid": 0, "block": 0})
        return (out, torch.zeros((0, 0), dtype=torch.uint8, device=q.device)) if record_visits else out

    # (a table that had to be copied, or is looked at on every call, is not repeated from a record)
    keeps = key is not None and kt is k_table and vt is v_table and out.data_ptr() % 16 == 0 and \
        _env("LOOPFUSE_CHECK_TABLES", "0") != "1"
    P.q, P.k, P.v, P.o = q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr()
    P.k_table = kt.data_ptr() if kt is not None else None
    P.v_table = vt.data_ptr() if vt is not None else None
    P.B, P.Hq, P.Hkv, P.Sq, P.Sk = B, Hq, Hkv, Sq, Sk
    P.window = int(plan.window)
    P.scale = float(plan.scale)
    P.softcap = softcap if softcap is not None else 0.0
    P.denom_add = float(plan.denom_add)
    if plan.denom_add < 0.0 or not math.isfinite(plan.denom_add):
        raise UnsupportedPlan("the denominator offset must be finite and >= 0")
    P.nsplit, P.rows, P.split_len = 1, 1, 0

    # ---- additive biases: [B, Hq, Sq, X] views with broadcast (stride 0) batch/head/row dims
    bias_bits = 0

    def bias_layout(t: torch.Tensor, what: str, last: int):
        nonlocal bias_bits
        if t.dtype != dtype or not t.is_cuda:
            raise UnsupportedPlan(f"{what} must be a {dtype} GPU tensor")
        if t.dim() > 4:
            raise UnsupportedPlan(f"{what} has more than 4 dims")
        if _env("LOOPFUSE_BIAS_COPY", "1") == "1" and \
                t.dim() >= 2 and t.shape[-1] == last and t.stride(-1) == 1 and t.numel() <= (1 << 25) and \
                (t.data_ptr() % 8 or any(st % 4 for n, st in zip(t.shape[:-1], t.stride()[:-1]) if n > 1)):
            # rows that do not start on 8-byte borders (a mask over an odd number of keys) would
            # be read element by element: a copy with padded rows is cheaper for tensors this small
            padded = torch.empty((*t.shape[:-1], (last + 3) // 4 * 4), dtype=t.dtype, device=t.device)
            t = padded[..., :last].copy_(t)
        try:
            t = t.expand(B, Hq, Sq, last)
        except RuntimeError:
            raise UnsupportedPlan(f"{what} does not broadcast to [{B}, {Hq}, {Sq}, {last}]")
        if t.stride(3) != 1 and t.shape[3] != 1:
            raise UnsupportedPlan(f"{what} needs last-dim stride 1")
        if t.data_ptr() % 8 or any(st % 4 for n, st in zip(t.shape[:3], t.stride()[:3]) if n > 1):
            bias_bits |= 4          # rows not 8-byte aligned: element loads
        return t

    if score_bias is not None:
        score_bias = bias_layout(score_bias, "score bias", Sk)
        P.bias = score_bias.data_ptr()
        P.bias_sb, P.bias_sh, P.bias_sq = score_bias.stride(0), score_bias.stride(1), score_bias.stride(2)
        bias_bits |= 1
    mask_own = None        # the mask without the dims it is shared over, while nothing of it is written yet
    if score_mask is not None:
        if score_bias is not None:
            raise UnsupportedPlan("a score mask and a score bias")
        if score_mask.dtype != torch.bool:
            raise UnsupportedPlan("the score mask must be a boolean tensor")
        try:
            score_mask = score_mask.expand(B, Hq, Sq, Sk)
        except RuntimeError:
            raise UnsupportedPlan(f"score mask does not broadcast to [{B}, {Hq}, {Sq}, {Sk}]")
        mask_own = score_mask[tuple(slice(0, 1) if st == 0 else slice(None) for st in score_mask.stride()[:3])]
        P.bias_sb, P.bias_sh, P.bias_sq = (int(st != 0) for st in score_mask.stride()[:3])      # what it is shared over; strides below
        bias_bits |= 1

    def write_mask_bias():
        """The whole bias of a boolean mask, for the kernels that read every element of it."""
        nonlocal mask_own, score_bias
        if mask_own is not None:
            shown, hidden = 0.0, float("-inf")
            mask_buf = torch.empty((*mask_own.shape[:3], (Sk + 7) // 8 * 8), dtype=dtype, device=q.device)[..., :Sk]
            mask_buf.fill_(hidden if mask_keep else shown).masked_fill_(mask_own, shown if mask_keep else hidden)
            score_bias = mask_buf.expand(B, Hq, Sq, Sk)
            P.bias = mask_buf.data_ptr()
            P.bias_sb, P.bias_sh, P.bias_sq = score_bias.stride(0), score_bias.stride(1), score_bias.stride(2)
            mask_own = None

    if out_bias is not None:
        out_bias = bias_layout(out_bias, "output bias", D)
        P.obias = out_bias.data_ptr()
        P.ob_sb, P.ob_sh, P.ob_sq = out_bias.stride(0), out_bias.stride(1), out_bias.stride(2)
        bias_bits |= 2
    d2 = 0
    if (q2 is None) != (k2 is None):
        raise UnsupportedPlan("q2 and k2 come together")
    if q2 is not None:
        if q2.dim() != 4 or k2.dim() != 4 or q2.shape[:3] != (B, Hq, Sq):
            raise UnsupportedPlan(f"Q2 must be [{B}, {Hq}, {Sq}, D2]")
        d2 = q2.shape[3]
        if d2 not in (16, 32, 64):
            raise UnsupportedPlan(f"depth {d2} of the second score product not supported (16, 32, 64)")
        if k2.shape[0] != B or k2.shape[2] != Sk or k2.shape[3] != d2 or k2.shape[1] < 1 or Hq % k2.shape[1]:
            raise UnsupportedPlan(f"K2 must be [{B}, H2 | {Hq}, {Sk}, {d2}]")
        _check_tensor("Q2", q2, dtype)
        _check_tensor("K2", k2, dtype)
        P.q2, P.k2 = q2.data_ptr(), k2.data_ptr()
        P.q2_sb, P.q2_sh, P.q2_ss = q2.stride(0), q2.stride(1), q2.stride(2)
        P.k2_sb, P.k2_sh, P.k2_ss = k2.stride(0), k2.stride(1), k2.stride(2)
        P.k2_group = Hq // k2.shape[1]
    if bias_bits not in (0, 1) or plan.denom_add != 0.0 or d2:
        force_family = "prefill"       # the decode kernel takes an aligned score bias and nothing else of these

    # ---- family: decode when there is no mask and few query rows share a KV head
    family = force_family
    if family is None:
        few = (Sq == 1 and group <= 64) or (group == 1 and Sq <= 16)
        # a caller that wants the row log-sum-exp (a forward that a backward will follow) gets the
        # prefill kernel, which writes it; the decode kernels do not
        family = "decode" if (mask == MASK_NONE and few and Sk >= 16 and lse is None) else "prefill"
    keep = (q, k, v, out, kt, vt, score_bias, score_mask, out_bias, q2, k2)  # noqa: F841  (tensors stay alive until the launch is queued)

    if family == "prefill" and not bias_bits and plan.denom_add == 0.0 and not d2:
        family = {"swp": "prefill_swp", "w32": "prefill"}.get(choice.get("prefill"), None) or prefill_variant(Sq, v_tr)
    # a score bias with 8-byte aligned rows and nothing else special: the direct-to-LDS kernel with the bias
    # classified tile by tile first (lf_bias_classify) -- what a mask given as a tensor needs
    bias_tiles = (family == "prefill" and bias_bits == 1 and plan.denom_add == 0.0 and not d2
                  and lse is None and Sk >= 4 and (Sk + 63) // 64 <= 65535 * 4 and B * Hq <= 65535
                  and _env("LOOPFUSE_BIAS_TILES", "1") == "1" and choice.get("prefill") != "w32"
                  and prefill_variant(Sq, v_tr) == "prefill_swp")
    if bias_tiles:
        family = "prefill_swp"
    if family == "prefill_swp":
        # direct-to-LDS staging addresses memory with 32-bit byte offsets.  Dense operands:
        # offsets inside one (batch, kv head) span; the kernel also addresses up to three
        # tiles past Sk (those reads are range-checked to zeros, but their offsets must
        # not wrap).  Paged operands: offsets inside the whole pool (< 4 GiB), pages of a
        # multiple of 8 tokens (the rows of one wave-level load stay inside a page).
        def swp_ok(t, is_paged, ps_, ss):
            if is_paged:
                span_b = 2 * (sum((n - 1) * abs(st) for n, st in zip(t.shape, t.stride())) + 1)
                return ps_ % 8 == 0 and span_b < (1 << 32) - 64 and all(st >= 0 for st in t.stride())
            reach = abs(ss) * 2 * (Sk + 3 * 64) + 2 * D
            return ss >= 0 and reach < (1 << 32) and (Sk - 1) * abs(ss) * 2 + 2 * D < (1 << 31)
        if not (swp_ok(k, plan.k_paged, page_size, P.k_ss)
                and swp_ok(v, plan.v_paged, page_size_v or page_size, P.v_ss)) \
                or (paged and _env("LOOPFUSE_PAGED_SWP", "1") != "1"):
            family = "prefill"
        if plan.k_paged:
            P.k_span = sum((n - 1) * st for n, st in zip(k.shape, k.stride())) + 1
        if plan.v_paged:
            P.v_span = sum((n - 1) * st for n, st in zip(v.shape, v.stride())) + 1
    if family in ("prefill", "prefill_swp"):
        P.q_sb, P.q_sh, P.q_ss = q.stride(0), q.stride(1), q.stride(2)
        P.o_sb, P.o_sh, P.o_ss = out.stride(0), out.stride(1), out.stride(2)
        extra = tuple(_env("LOOPFUSE_KOPTS", "").split())
        # buffer loads address a (batch, kv head) span with 32-bit byte offsets
        span = max((Sk - 1) * abs(P.k_ss), (Sk - 1) * abs(P.v_ss)) * 2 + 2 * D
        if family == "prefill" and span >= (1 << 31):
            extra += ("-DLF_KVBUF=0",)
        elif family == "prefill" and (bias_bits or d2) and not paged:
            extra += ("-DLF_DMA=1",)     # frees the staging registers the bias values / Q2 fragments need
        # grouped-query attention: the 4 waves of a workgroup take 4 (or 2) query heads of one
        # group over the same query rows and share every K/V tile in LDS
        pack = 0
        if family == "prefill_swp" and group % 2 == 0 and not any(e.startswith("-DLF_NW=") for e in extra) and \
                choice.get("pack", _env("LOOPFUSE_GQAPACK", "1") == "1") and (not bias_bits or P.bias_sh == 0):
            # (with a score bias only when all heads share it: the tile classes are then the same for the
            # packed heads of a workgroup)
            pack = 4 if group % 4 == 0 else 2
        if family == "prefill_swp" and bias_bits and not bias_tiles:
            family = "prefill"                          # swp was refused above (spans): the register-staged kernel
        if family != "prefill_swp" or (mask_own is not None and mask_own.stride(3) != 1):
            write_mask_bias()
            keep += (score_bias,)
        if mask_own is not None:
            bias_bits = MASK_BITS
        spec = _spec(family, _DTYPE_CODE[dtype], D, mask, plan.softcap is not None, paged,
                     page_size, table_i64, v_tr=v_tr if family == "prefill" else True, bias=bias_bits,
                     denom=plan.denom_add != 0.0, d2=d2, page_size_v=page_size_v, pack=pack, extra=extra,
                     safe=plan.zero_blind_rows and bool(bias_bits & (1 | MASK_BITS)),
                     bn=prefill_kv_tile(D, bias_bits, choice, B * (Hq // (pack or 1)) * (-(-Sq // (128 // (pack or 1)))),
                                        min(Sk, P.window) if mask == MASK_SLIDING else Sk)
                     if family == "prefill_swp" else 0,
                     stay=family == "prefill_swp" and prefill_out_stays(2 * B * Hq * Sq * D))
        bm, bn = TILE_SHAPES[family]
        nw = 4
        for e in spec.extra:                    # tuning: -DLF_NW=8 doubles the q tile
            if e.startswith("-DLF_NW="):
                nw = int(e.split("=")[1])
                bm = 32 * nw
        if spec.bn:
            bn = spec.bn
        heads = Hq
        if spec.pack:
            bm, heads = 128 // spec.pack, Hq // spec.pack      # q tiles of 32 rows x 4 heads, or 64 rows x 2 heads
        nqt = (Sq + bm - 1) // bm
        nkt = (Sk + bn - 1) // bn
        visits = None
        if record_visits:
            visits = torch.zeros((B * heads * nqt, nkt), dtype=torch.uint8, device=q.device)
            P.visits = visits.data_ptr()
        # lf_attn_prefill_swp: one q tile per workgroup; lf_attn_prefill: two (a long and a short one)
        grid = xcd_slots(B * heads, nqt if family == "prefill_swp" else (nqt + 1) // 2)
        if lse is not None:
            if family != "prefill_swp" or paged:
                raise UnsupportedPlan("the row log-sum-exp is written by lf_attn_prefill_swp for dense K/V only")
            if lse.dtype != torch.float32 or tuple(lse.shape) != (B, Hq, Sq) or not lse.is_contiguous() or lse.device != q.device:
                raise UnsupportedPlan(f"lse must be a contiguous float32 [{B}, {Hq}, {Sq}] tensor on the device of Q")
            P.part_ml = lse.data_ptr()
        names = [spec.entry()]
        if family == "prefill_swp" and bias_bits:
            nb_, nh_ = (B if P.bias_sb else 1), (Hq if P.bias_sh else 1)
            if mask_own is not None:
                # the mask's bits and the words of its 32 x 32 blocks, once per distinct (batch, head) it holds
                classify, nrb, chunks = "lf_mask_tiles", (-(-Sq // 32) if P.bias_sq else 1), -(-Sk // 1024)
                words = nb_ * nh_ * nrb * chunks
                table = torch.empty((words + nb_ * nh_ * nrb * -(-Sk // 32) * 16,), dtype=torch.int64, device=q.device)
                P.part_acc, P.bias = table.data_ptr(), table.data_ptr() + 8 * words
                P.obias, P.rows = mask_own.data_ptr(), int(mask_keep)
                P.ob_sb, P.ob_sh, P.ob_sq = (st if n > 1 else 0 for n, st in zip(mask_own.shape, mask_own.stride()[:3]))
                ahead = (nrb, nb_ * nh_, chunks)
            else:
                # tile classes of the bias, once per distinct (batch, head) it holds: int32 [units][kv tiles]
                classify, ahead = "lf_bias_classify", (nqt, nb_ * nh_, (nkt + 3) // 4)
                table = torch.empty((nb_ * nh_ * nqt * nkt,), dtype=torch.int32, device=q.device)
                P.part_acc = table.data_ptr()
            keep += (table,)
            get_kernel(spec, classify).launch(ahead, (256, 1, 1), P)
            names.insert(0, classify)
        fn = get_kernel(spec, spec.entry())
        record = {"kernels": names, "grid": grid, "block": 64 * nw, "q_tile_rows": bm, "kv_tile_rows": bn,
                  "heads_per_workgroup": spec.pack or 1}
        if keeps:
            kept = _Kept(P, [(fn, (grid, 1, 1), 64 * nw)], ((B, Hq, Sq, D), dtype), record)
            kept.launches.launch(P)
            _keep(key, kept)
        else:
            fn.launch((grid, 1, 1), (64 * nw, 1, 1), P)
        _last_launch.set(dict(record))
        return (out, visits) if record_visits else out

    if family != "decode":
        raise ValueError(f"unknown kernel family {family!r}")
    if lse is not None:
        raise UnsupportedPlan("the decode kernels do not write the row log-sum-exp")
    if mask != MASK_NONE:
        raise UnsupportedPlan("the decode kernel takes no mask")
    write_mask_bias()
    # query rows of one unit: the group's heads (Sq == 1) or the Sq rows (group == 1)
    if Sq == 1:
        rows = group
        P.q_sb, P.q_sh, P.q_ss = q.stride(0), group * q.stride(1), q.stride(1)
        P.o_sb, P.o_sh, P.o_ss = out.stride(0), group * out.stride(1), out.stride(1)
        if bias_bits:
            P.bias_sh, P.bias_sq = group * score_bias.stride(1), score_bias.stride(1)
    elif group == 1:
        rows = Sq
        P.q_sb, P.q_sh, P.q_ss = q.stride(0), q.stride(1), q.stride(2)
        P.o_sb, P.o_sh, P.o_ss = out.stride(0), out.stride(1), out.stride(2)
    else:
        raise UnsupportedPlan("decode needs Sq == 1 or group == 1")
    chunks = (rows + DECODE_QROWS - 1) // DECODE_QROWS
    units = B * Hkv * chunks
    waves = int(_env("LOOPFUSE_DECODE_WAVES", "4"))
    # Token-major page pools ([pages, page, Hkv, D]: the heads of a token side by side)
    # are read whole-page-wise when the 8 waves of a workgroup take 8 consecutive heads.
    coop = _decode_coop_waves(paged, page_size, page_size_v, bias_bits, Hkv, P, D)
    if "head_per_wave" in choice:
        headwave = bool(choice["head_per_wave"]) and paged == 3 and (Hkv % 8 == 0 or coop > 0)
    elif not coop or _env("LOOPFUSE_DECODE_HEADWAVE") is not None:
        headwave = _decode_headwave(paged, page_size, Hkv, D, P, B * ((Hkv + 7) // 8) * chunks, Sk) and not page_size_v
    else:
        units_coop = B * (Hkv // coop) * chunks
        if static_scratch:
            headwave = decode_coop_pays(units_coop, Sk, min(rows, DECODE_QROWS), page_size)
            if not (headwave or num_splits or choice.get("splits")) and decode_coop_fills(units_coop, Sk, page_size):
                # more splits of fewer workgroups: a step that does not run in the static array with the other loads may with these
                headwave = not static_split_runs(decode_split(units, Sk), Sk, B * Hkv * rows, D, runtime.static_scratch_bytes())
        elif _env("LOOPFUSE_DECODE_SPLITS") or num_splits or choice.get("splits"):
            headwave = decode_coop_pays(units_coop, Sk, min(rows, DECODE_QROWS), page_size)      # (a given count: neither rule's)
        else:
            headwave = decode_coop_beats(units_coop, coop, units, Sk, min(rows, DECODE_QROWS), page_size, D)
    coop = coop if headwave else 0
    if headwave:
        waves = coop or 8
        units = B * ((Hkv + waves - 1) // waves) * chunks
    num_splits = num_splits or choice.get("splits")
    if not num_splits and coop:
        num_splits = decode_coop_split(units, Sk, min(rows, DECODE_QROWS))
        if static_scratch:
            eight = bool(choice["head_per_wave"]) and Hkv % 8 == 0 if "head_per_wave" in choice else \
                _decode_headwave(paged, page_size, Hkv, D, P, B * ((Hkv + 7) // 8) * chunks, Sk)
            plain = decode_split(B * ((Hkv + 7) // 8 if eight else Hkv) * chunks, Sk, per_cu=1 if eight else 2)
            num_splits = decode_static_split(num_splits, plain, Sk, B * Hkv * rows, D, runtime.static_scratch_bytes())
    elif not num_splits and (headwave or static_scratch or _env("LOOPFUSE_DECODE_SPLITS")):
        num_splits = decode_split(units, Sk, per_cu=1 if headwave else 2)
    elif not num_splits:
        num_splits = decode_even_split(units, Sk, D, rows=B * Hkv * rows)
    nsplit, split_len = _split_lengths(num_splits, Sk)
    P.rows, P.nsplit, P.split_len = rows, nsplit, split_len
    spec = _spec("decode", _DTYPE_CODE[dtype], D, MASK_NONE, plan.softcap is not None, paged,
                 page_size, table_i64, rows=DECODE_QROWS, waves=waves, headwave=headwave, page_size_v=page_size_v,
                 coop=coop > 0,
                 rowload=not coop and _decode_rowload(paged, page_size, page_size_v, bias_bits),
                 bias=bias_bits, safe=plan.zero_blind_rows and bool(bias_bits),
                 extra=tuple(_env("LOOPFUSE_KOPTS", "").split()))
    combine_grid = decode_combine_grid(B * Hkv * rows, nsplit, D)
    if static_scratch:
        if nsplit <= 1 or not merge_splits:
            raise UnsupportedPlan("static_scratch serves split decode steps (this call does not split the keys)")
        nrow = B * Hkv * rows * nsplit
        runtime.launch_decode_static(get_kernel(spec, "lf_attn_decode"), get_kernel(spec, "lf_attn_decode_combine"), P,
                                     4 * nrow * D, 4 * nrow * 2, (units, nsplit), 64 * spec.waves, combine_grid, 256)
        _last_launch.set({"kernels": ["lf_attn_decode", "lf_attn_decode_combine"], "grid": (units, nsplit),
                                 "block": 64 * spec.waves, "head_per_wave": headwave, "cooperative_loads": spec.coop,
                                 "static_scratch": True})
        return out
    named = _kernels_of(spec)
    step, combine = get_kernel(spec, "lf_attn_decode", named), get_kernel(spec, "lf_attn_decode_combine", named)
    steps = [(step, (units, nsplit, 1), 64 * spec.waves)] + ([(combine, (combine_grid, 1, 1), 256)] if nsplit > 1 else [])
    record = {"kernels": ["lf_attn_decode"] + (["lf_attn_decode_combine"] if nsplit > 1 and merge_splits else []),
              "grid": (units, nsplit), "block": 64 * spec.waves, "head_per_wave": headwave,
              "cooperative_loads": spec.coop}
    nrow = B * Hkv * rows * nsplit
    if keeps:
        kept = _Kept(P, steps, ((B, Hq, Sq, D), dtype), record, (nrow * (D + 2), 4 * nrow * D) if nsplit > 1 else None)
    if nsplit > 1:
        with _scratch_lock:        # no other thread's step on this stream between the two launches
            scratch = _get_scratch(q.device, nrow * (D + 2))
            P.part_acc = scratch.data_ptr()
            P.part_ml = scratch.data_ptr() + 4 * nrow * D
            if keeps:
                kept.launches.launch(P)
            else:
                step.launch((units, nsplit, 1), (64 * spec.waves, 1, 1), P)
                if merge_splits:
                    combine.launch((combine_grid, 1, 1), (256, 1, 1), P)
    elif keeps:
        kept.launches.launch(P)
    else:
        step.launch((units, nsplit, 1), (64 * spec.waves, 1, 1), P)
    if keeps:
        _keep(key, kept)
    _last_launch.set(dict(record))
    return out


# ---------------------------------------------------------------------------
# backward (the reference has none: loopfuse README "future work")
# ---------------------------------------------------------------------------
class AttnBwdParams(ctypes.Structure):
    """Mirror of ``struct LfAttnBwdParams`` in csrc/kernels/lf_attn_bwd.hip."""

    _fields_ = (
        [(n, ctypes.c_void_p) for n in ("q", "k", "v", "o", "dout", "dq", "dk", "dv", "lse", "delta")]
        + [(f"{t}_{x}", ctypes.c_longlong) for t in ("q", "k", "v", "o", "do", "dq", "dk", "dv") for x in ("sb", "sh", "ss")]
        + [(n, ctypes.c_int) for n in ("B", "Hq", "Hkv", "Sq", "Sk", "window")]
        + [("scale", ctypes.c_float), ("softcap", ctypes.c_float), ("ds", ctypes.c_void_p), ("ds_sh", ctypes.c_longlong)]
    )


BWD_DS_BLOCK = 32 * 32      # elements of a block of dS (lf_bw_ds_row in csrc/kernels/lf_attn_bwd.hip)


def bwd_q_split(D: int, mask: int, units: int, Sk: int) -> bool:
    """Is lf_attn_bwd_dkdv launched with workgroups of 64 keys, whose waves hold each 32 of them twice, one for the first and one
    for the last 32 queries of a tile?  Twice the workgroups and half as long a chain of tiles in each, against twice the Q / dO
    loads: it pays where the workgroups of 128 keys leave CUs idle, or alone with the longest of them.  ``units`` = batch x
    kv heads.  All launches, whole / split, us, over 70 shapes: causal D 64 B8 16/4 S1000 (256 workgroups of 128 keys) 140 / 110,
    B10 64/8 S445 (320) 170 / 126, B5 16/4 S3539 (560) 607 / 614; causal D 128 B1 32/8 S2048 (128) 307 / 209, B6 H8 S500 (192)
    44.6 / 44.6, B10 8/2 S1748 (280) 328 / 367; window D 64 B3 8/4 S2183 (216) 91 / 76, B15 64/8 S383 (360) 148 / 136, B6 16/2
    S5110 (480) 267 / 277, D 128 B2 64/8 S524 (80) 97 / 66, B3 32/8 S1055 (216) 106 / 113; unmasked D 64 B1 16/8 S2120 (136)
    155 / 135, B1 H8 S5043 (320) 279 / 280, D 128 B6 H4 S1784 (336) 177 / 170, B10 H4 S1879 (600) 320 / 326."""
    n = units * -(-Sk // 128)
    if mask == MASK_NONE:
        return n <= (192 if D == 64 else 352)
    return n <= (384 if D == 64 else 192)


def bwd_ds_blocks(mask: int, window: int, Sq: int, Sk: int) -> int:
    """Blocks of dS of one (batch, query head): ``lf_bw_ds_row`` of the row behind the last, and under a window the blocks in
    front of the first key that the last row's start leaves out."""
    nqb, nkb = -(-Sq // 32), -(-Sk // 32)
    if mask == MASK_NONE:
        return nqb * nkb
    if mask == MASK_CAUSAL:
        m = min(nqb, nkb)
        return m * (m + 1) // 2 + (nqb - m) * nkb
    return nqb * ((window + 30) // 32 + 1)


def bwd_dq_threads(D: int, mask: int, softcap: bool, units: int, Sq: int, Sk: int) -> int:
    """Workgroup size of lf_attn_bwd_dq: 512 (256 query rows, two waves per SIMD on one K/V tile stream) or 256 (128 rows,
    twice the workgroups).  ``units`` = batch x query heads.  Head dimension 128: a CU's LDS holds one workgroup of either,
    so the larger one wins once all CUs have work -- more than 128 of them, and more than 256 under a causal mask, where
    the longest q tile is the launch: 512 against 256 threads, us, causal 64 workgroups 74 / 57, 256 80 / 71, 384 61 / 73,
    1024 233 / 294; unmasked 64 77 / 59, 192 157 / 218; window 256: 64 25 / 18, 192 28 / 38, 1024 112 / 144.  Head
    dimension 64: two workgroups of 256 threads fit and balance better (B16 32/8 S300 41 / 32, window 256 B4 H32 S2048
    71 / 62) except over long sequences, where halving the K/V traffic counts (causal B2 H16 S4096 121 / 133)."""
    n = units * -(-Sq // 256)
    if n <= (256 if mask == MASK_CAUSAL else 128) or (D == 64 and (Sk < 4096 or softcap or mask == MASK_SLIDING)):
        return 256
    return 512


def bwd_two_key_blocks(D: int, mask: int, softcap: bool) -> bool:
    """Is lf_attn_bwd_dkdv built with two key blocks per wave?  Its accumulators are right only while the compiler leaves
    them where they are, so the forms that are built are those whose code is checked; beside the values of a window or a
    softcap two blocks leave it next to no registers, and gain nothing."""
    return D == 128 and not softcap and mask != MASK_SLIDING


def bwd_key_blocks(D: int, mask: int, softcap: bool, units: int, Sk: int) -> int:
    """32-key blocks a wave of lf_attn_bwd_dkdv holds: 2 (workgroups of 256 keys; every fragment read from
    LDS feeds two MFMAs) or 1 (128 keys).  ``units`` = batch x kv heads.  Measured, all backward launches, 2 against 1:
    causal B4 H32 S2048 541 / 570 us, B2 H32 S4096 946 / 1005 us, unmasked 6 % faster throughout, but the launch has to
    stay balanced: causal with 256 such workgroups 1.13 ... 1.21 times slower (one long key block per CU), 512 of them at
    S 1024 1.07 times, unmasked with a last round that is nearly empty (280 workgroups) 1.07 times.  A sliding window walks
    more blocks than its waves need (0.95 ... 1.08 times), head dimension 64 runs two workgroups per CU with one block
    (1.03 ... 1.3 times), and a softcap's values do not fit the registers beside two."""
    n = units * -(-Sk // 256)
    if not bwd_two_key_blocks(D, mask, softcap):
        return 1
    if mask == MASK_CAUSAL:
        return 2 if (n >= 512 and Sk >= 2048) or (n >= 1024 and Sk >= 1024) else 1
    return 2 if n >= 256 and n >= 0.85 * 256 * -(-n // 256) else 1


def bwd_keep_ds(D: int, softcap: bool, units: int, group: int, Sk: int, blocks: int) -> bool:
    """Does lf_attn_bwd_dkdv leave dS in memory, so that lf_attn_bwd_dq is one product that reads it instead of three that form
    it again?  ``units`` = batch x query heads, ``blocks`` = of dS in all (2 KB each; up to 2 GiB).  Seven products instead of
    nine against 2 bytes per visible score written and read, both by non-temporal accesses.  All launches, recomputed / kept, us:
    head dimension 128, causal B4 H32 S2048 549 / 521 (545 MB), B2 32/8 S4096 953 / 909, B6 64/32 S769 369 / 307, with a softcap
    B4 32/8 S2048 644 / 561, window 256 252 / 204, unmasked H2 S7033 392 / 311; of 60 drawn shapes three were slower by more than
    2 %, short ones with eight heads per group (B6 16/2 S135 62 / 65).  Head dimension 64 has half the matrix work per score:
    with a softcap B4 H32 S2048 424 / 379, without B4 H32 S2048 304 / 333, B8 16/4 S1000 140 / 143, and kept where few heads leave
    CUs to the recomputation's longest workgroups: H8 S4520 181 / 158, H2 S1038 52 / 47, B4 H16 S535 50 / 47."""
    size = 2 * BWD_DS_BLOCK * blocks
    if size > 2 << 30 or (Sk < 192 and group > 4):
        return False
    return D == 128 or softcap or (units <= 64 and group <= 4 and Sk >= 512 and size <= 176 << 20)


def bwd_grads_stay(nbytes: int) -> bool:
    """Are the gradients written by plain stores (``-DLF_STAY=1``), which leave them near whoever reads them next, and not in
    whole rows past the caches?  ``nbytes`` = size of dQ.  Whole over plain, 57 shapes, all launches alone / with an element-wise kernel
    behind them that reads the gradients: below 10 MB 0.98 ... 1.04 / 0.99 ... 1.13, 10 ... 30 MB 0.95 ... 1.00 / 0.99 ... 1.03,
    above 0.90 ... 1.00 / 0.95 ... 1.01."""
    return nbytes < 10_000_000


@functools.lru_cache(maxsize=512)
def bwd_spec(dtype: torch.dtype, D: int, mask: int, softcap: bool = False, key_blocks: int = 1,
             dq_threads: int = 512, keep_ds: bool = False, q_split: bool = False, stay: bool = False) -> KernelSpec:
    return KernelSpec("bwd", _DTYPE_CODE[dtype], D, mask, softcap, stay=stay,
                      extra=(f"-DLF_BW_DQ_NT={dq_threads}", f"-DLF_BW_W={key_blocks}") + (("-DLF_BW_DS=1",) if keep_ds else ())
                      + (("-DLF_BW_QSPLIT=1",) if q_split else ()))


def attention_backward(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, o: torch.Tensor, lse: torch.Tensor,
                       dout: torch.Tensor, plan: AttnPlan, *, key_blocks: Optional[int] = None,
                       dq_threads: Optional[int] = None, keep_ds: Optional[bool] = None, q_split: Optional[bool] = None):
    """Gradients of ``attention(q, k, v, plan)`` for dense K/V (mask none / causal / sliding, scale,
    softcap; no bias or paging): returns ``(dq, dk, dv)`` in the operands' dtype.  ``o`` and ``lse``
    are the forward's output and row log-sum-exp (``attention(..., lse=...)``).  Two or
    three launches (csrc/kernels/lf_attn_bwd.hip): delta = rowsum(dO * O), together with dQ where that has small
    workgroups and forms dS itself; dK and dV, one workgroup per 128 or 256 keys of a (batch, kv head); dQ, one workgroup per 128
    or 256 query rows, from dS left in a scratch tensor where ``bwd_keep_ds`` says so (``keep_ds`` overrides it).  No
    atomics: results are reproducible bit for bit.  ``key_blocks``, ``dq_threads`` and ``q_split`` override the rules of the work
    splits (``bwd_key_blocks``, ``bwd_dq_threads``, ``bwd_q_split``)."""
    given = key_blocks is not None or dq_threads is not None or keep_ds is not None or q_split is not None
    key = _signature("bwd", (q, k, v, o, lse, dout), plan,
                     {"key_blocks": key_blocks, "dq_threads": dq_threads, "keep_ds": keep_ds, "q_split": q_split} if given else None)
    kept = _kept.get(key)
    if kept is not None and kept.calls is not None:
        kept.calls -= 1
        if kept.calls < 0:
            kept = None
    room = True
    if kept is not None:
        res = _backward_again(kept, q, k, v, o, lse, dout)
        if res is not None:
            return res
        room = False                     # (dS asked for by the caller is tried again below, and its error raised)
    dtype = q.dtype
    if dtype not in _DTYPE_CODE:
        raise UnsupportedPlan(f"dtype {dtype} not supported by the MFMA kernels (bf16/fp16 only)")
    if plan.k_paged or plan.v_paged or plan.denom_add != 0.0:
        raise UnsupportedPlan("the backward kernels serve dense K/V and the plain softmax denominator")
    softcap = None
    if plan.softcap is not None:
        softcap = abs(float(plan.softcap))
        if not (softcap > 0.0) or not math.isfinite(softcap):
            raise UnsupportedPlan("softcap must be finite and non-zero")
    if q.dim() != 4 or k.dim() != 4 or v.dim() != 4:
        raise UnsupportedPlan("Q, K, V must be [B, H, S, D]")
    B, Hq, Sq, D = q.shape
    Hkv, Sk = k.shape[1], k.shape[2]
    if D not in (64, 128) or k.shape != v.shape or k.shape[0] != B or k.shape[3] != D or Hkv < 1 or Hq % Hkv:
        raise UnsupportedPlan(f"shapes not served: Q {tuple(q.shape)}, K {tuple(k.shape)}, V {tuple(v.shape)}")
    if Sq < 1 or Sk < 1:
        raise UnsupportedPlan("empty sequences")
    if o.shape != q.shape or dout.shape != q.shape or tuple(lse.shape) != (B, Hq, Sq):
        raise UnsupportedPlan("O, dO must have the shape of Q and lse must be [B, Hq, Sq]")
    if lse.dtype != torch.float32 or not lse.is_contiguous():
        raise UnsupportedPlan("lse must be contiguous float32")
    mask = {None: MASK_NONE, "none": MASK_NONE, "causal": MASK_CAUSAL, "sliding": MASK_SLIDING}.get(plan.mask)
    if mask is None:
        raise UnsupportedPlan(f"mask {plan.mask!r} not served")
    window = int(plan.window or 0)
    if mask == MASK_SLIDING and window < 1:
        raise UnsupportedPlan("sliding window must be >= 1")
    cap = softcap is not None
    if key_blocks and key_blocks != 1 and (key_blocks != 2 or not bwd_two_key_blocks(D, mask, cap)):
        raise UnsupportedPlan(f"key_blocks {key_blocks!r}: 1, or 2 at head dim 128 without a window and a softcap")
    if q_split and key_blocks and key_blocks != 1:
        raise UnsupportedPlan("q_split: with one key block per wave")
    if dq_threads and dq_threads not in (256, 512):
        raise UnsupportedPlan(f"dq_threads {dq_threads!r}: 256 or 512")
    for name, t in (("Q", q), ("K", k), ("V", v), ("O", o), ("dO", dout)):
        _check_tensor(name, t, dtype)
    # the tiles travel global -> LDS with 32-bit byte offsets inside one (batch, head) span, rows
    # past the end addressed too (and range-checked to zeros)
    for name, t, S in (("Q", q, Sq), ("dO", dout, Sq), ("K", k, Sk), ("V", v, Sk)):
        if t.stride(2) < D or (S + 64) * t.stride(2) * 2 + 2 * D >= (1 << 32):
            raise UnsupportedPlan(f"{name}: row stride {t.stride(2)} not served by the backward kernels' direct loads")
    dq = torch.empty((B, Hq, Sq, D), dtype=dtype, device=q.device)
    dk = torch.empty((B, Hkv, Sk, D), dtype=dtype, device=q.device)
    dv = torch.empty((B, Hkv, Sk, D), dtype=dtype, device=q.device)
    delta = torch.empty((B, Hq, Sq), dtype=torch.float32, device=q.device)
    P = AttnBwdParams()
    for name, t in (("q", q), ("k", k), ("v", v), ("o", o), ("dout", dout), ("dq", dq), ("dk", dk), ("dv", dv),
                    ("lse", lse), ("delta", delta)):
        setattr(P, name, t.data_ptr())
    P.q_sb, P.q_sh, P.q_ss = q.stride()[:3]
    P.k_sb, P.k_sh, P.k_ss = k.stride()[:3]
    P.v_sb, P.v_sh, P.v_ss = v.stride()[:3]
    P.o_sb, P.o_sh, P.o_ss = o.stride()[:3]
    P.do_sb, P.do_sh, P.do_ss = dout.stride()[:3]
    P.dq_sb, P.dq_sh, P.dq_ss = dq.stride()[:3]
    P.dk_sb, P.dk_sh, P.dk_ss = dk.stride()[:3]
    P.dv_sb, P.dv_sh, P.dv_ss = dv.stride()[:3]
    P.B, P.Hq, P.Hkv, P.Sq, P.Sk, P.window = B, Hq, Hkv, Sq, Sk, window
    P.scale = float(plan.scale)
    P.softcap = softcap if softcap is not None else 0.0
    keys = key_blocks or bwd_key_blocks(D, mask, cap, B * Hkv, Sk)
    nt = dq_threads or bwd_dq_threads(D, mask, cap, B * Hq, Sq, Sk)
    ds_blocks = bwd_ds_blocks(mask, window, Sq, Sk)
    ds = None
    if keep_ds or (keep_ds is None and room and bwd_keep_ds(D, cap, B * Hq, Hq // Hkv, Sk, B * Hq * ds_blocks)):
        try:
            ds = torch.empty((B * Hq, ds_blocks, BWD_DS_BLOCK), dtype=dtype, device=q.device)
            P.ds, P.ds_sh = ds.data_ptr(), ds.stride(0)
        except torch.OutOfMemoryError:
            if keep_ds:
                raise
            room = False                 # the gradients need no such room
    if q_split is None:
        q_split = not (key_blocks and key_blocks != 1) and bwd_q_split(D, mask, B * Hkv, Sk)
    if q_split:
        keys = 1
    spec = bwd_spec(dtype, D, mask, cap, keys, nt, ds is not None, q_split, bwd_grads_stay(2 * B * Hq * Sq * D))
    keep = (q, k, v, o, dout, lse, delta, dq, dk, dv, ds)  # noqa: F841  (tensors stay alive until the launches are queued)
    steps = {"lf_attn_bwd_delta": (-(-B * Hq * Sq // 16), 256),
             "lf_attn_bwd_dkdv": (xcd_slots(B * Hkv, -(-Sk // (128 * keys // (2 if q_split else 1)))), 256),
             "lf_attn_bwd_dq": (xcd_slots(B * Hkv, (Hq // Hkv) * -(-Sq // (nt // 2))), nt)}
    # without dS of lf_attn_bwd_dkdv, lf_attn_bwd_dq with 256 threads forms delta itself, and lf_attn_bwd_dkdv reads it
    names = ["lf_attn_bwd_dq", "lf_attn_bwd_dkdv"] if nt == 256 and ds is None else list(steps)
    named = _kernels_of(spec)
    launches = [(get_kernel(spec, name, named), (steps[name][0], 1, 1), steps[name][1]) for name in names]
    if key is not None:
        # An allocation that fails makes the allocator give back what it holds and wait for the device: the form without dS is
        # kept, and room for dS looked for again once in many calls
        kept = _Kept(P, launches, (dtype, None if ds is None else tuple(ds.shape)), {"kernels": names}, calls=None if room else _NO_ROOM_CALLS)
        kept.launches.launch(P)
        _keep(key, kept)
    else:
        for fn, grid, block in launches:
            fn.launch(grid, (block, 1, 1), P)
    _last_launch.set({"kernels": names})
    return dq, dk, dv


def _backward_again(kept: _Kept, q, k, v, o, lse, dout):
    """The launches of a signature seen before; None where there is no room for dS any more."""
    dtype, ds_shape = kept.results
    P = AttnBwdParams.from_buffer_copy(kept.params)
    dev = q.device
    dq, dk, dv = torch.empty(q.shape, dtype=dtype, device=dev), torch.empty(k.shape, dtype=dtype, device=dev), torch.empty(k.shape, dtype=dtype, device=dev)
    delta = torch.empty(lse.shape, dtype=torch.float32, device=dev)
    if ds_shape is not None:
        # last: it may take what room is left, which the results need and it does not
        try:
            ds = torch.empty(ds_shape, dtype=dtype, device=dev)
        except torch.OutOfMemoryError:
            return None
        P.ds = ds.data_ptr()
    P.q, P.k, P.v, P.o, P.dout = q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), dout.data_ptr()
    P.dq, P.dk, P.dv, P.lse, P.delta = dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), lse.data_ptr(), delta.data_ptr()
    kept.launches.launch(P)
    _last_launch.set(kept.record)
    return dq, dk, dv
