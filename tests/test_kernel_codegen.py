"""Static checks on the code objects of the kernels whose MFMAs are inline asm with explicit
register files (lf_attn_bwd_dkdv and lf_attn_bwd_dq, in every form that is built).

The compiler does not know the latency of those MFMAs: a register copy or a spill it decides
to place right behind one reads the accumulator before the result is there, and nothing at run
time says so.  The sources are written so that it has no reason to (every accumulator is pinned
to one register file, the live ranges fit), and this test holds the generated code to it:
compiled as the library compiles them (hipRTC, no GPU needed), disassembled, and checked for
  * no scratch-memory access at all (no spills),
  * every read of an MFMA's AGPR result by a non-MFMA instruction at least MIN_GAP
    instructions behind the MFMA that wrote it, or behind an explicit drain (s_nop >= 9),
  * no instruction other than the chain's own MFMAs touching the VGPR destination of an MFMA
    between that MFMA and the drain behind its chain,
  * no instruction but MFMAs touching an AGPR between the first and the last of them, and every MFMA with an AGPR
    destination naming the same tuple as its source: the accumulators are handed over as inputs there, so the compiler
    takes them for constants, and
  * two wait states between a vector instruction and an MFMA that reads what it wrote.
"""
import dataclasses
import os
import re
import shutil
import subprocess

import pytest
import torch

from loopfuse_amd import lowering, runtime

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
MIN_GAP = 24     # instructions; 12 wait states for the result plus one MFMA that may run ahead of it

pytestmark = pytest.mark.skipif(not os.path.exists(OBJDUMP) or shutil.which("hipcc") is None,
                                reason="needs the ROCm LLVM tools")


def _kernels(spec):
    code = lowering.compile_spec(spec).code_object
    path = os.path.join(os.environ.get("TMPDIR", "/tmp"), f"lf_codegen_{os.getpid()}.hsaco")
    with open(path, "wb") as fh:
        fh.write(code)
    try:
        text = subprocess.run([OBJDUMP, "-d", path], capture_output=True, text=True, check=True).stdout
    finally:
        os.unlink(path)
    parts = re.split(r"\n[0-9a-f]+ <(\w+)>:\n", text)
    out = {}
    for name, body in zip(parts[1::2], parts[2::2]):
        out[name] = [ln.split("//")[0].strip() for ln in body.splitlines() if ln.strip()]
    return out


def _check(name, lines):
    assert not [ln for ln in lines if ln.startswith("scratch_")], f"{name}: scratch memory accesses (spills)"
    mfma_dst = []           # (index, first, last) of MFMAs with an AGPR destination
    for i, ln in enumerate(lines):
        m = re.match(r"v_mfma_\S+ a\[(\d+):(\d+)\]", ln)
        if m:
            mfma_dst.append((i, int(m.group(1)), int(m.group(2))))
    for i, ln in enumerate(lines):
        m = re.match(r"v_accvgpr_read_b32 v\d+, a(\d+)", ln) or re.match(r"v_accvgpr_mov_b32 a\d+, a(\d+)", ln)
        if not m:
            continue
        reg = int(m.group(1))
        writers = [j for j, lo, hi in mfma_dst if j < i and lo <= reg <= hi]
        if not writers:
            continue
        j = writers[-1]
        between = lines[j + 1:i]
        drained = any(re.match(r"s_nop (\d+)", x) and int(re.match(r"s_nop (\d+)", x).group(1)) >= 9 for x in between)
        assert drained or len(between) >= MIN_GAP, \
            f"{name}: '{ln}' reads a{reg} {len(between)} instructions behind the MFMA that writes it ('{lines[j]}')"
    if not mfma_dst:
        return          # MFMAs issued through the builtin only: the compiler places their wait states itself
    # MFMAs with a VGPR destination (S^T / dP^T): until the drain behind the chain -- or MIN_GAP instructions --
    # nothing but the chain's own MFMAs may touch the destination registers (a copy or a live-range split the
    # compiler placed there would read or overwrite an accumulator that is not written yet)
    for j, ln in enumerate(lines):
        m = re.match(r"v_mfma_\S+ v\[(\d+):(\d+)\]", ln)
        if not m:
            continue
        lo, hi = int(m.group(1)), int(m.group(2))
        for gap, x in enumerate(lines[j + 1:j + 1 + MIN_GAP]):
            nop = re.match(r"s_nop (\d+)", x)
            if nop and int(nop.group(1)) >= 9:
                break
            if x.startswith("v_mfma"):
                continue
            regs = {int(r) for r in re.findall(r"\bv(\d+)\b", x)}
            for a, b in re.findall(r"\bv\[(\d+):(\d+)\]", x):
                regs.update(range(int(a), int(b) + 1))
            hit = sorted(r for r in regs if lo <= r <= hi)
            assert not hit, f"{name}: '{x}' touches v{hit[0]} {gap} instructions behind '{ln}', before its drain"


SPECS = [
    lowering.bwd_spec(torch.bfloat16, 128, lowering.MASK_CAUSAL),
    lowering.bwd_spec(torch.float16, 64, lowering.MASK_NONE),
    lowering.bwd_spec(torch.bfloat16, 128, lowering.MASK_SLIDING),     # 4-wave dQ kernel
    lowering.bwd_spec(torch.float16, 64, lowering.MASK_SLIDING),
    lowering.bwd_spec(torch.bfloat16, 128, lowering.MASK_CAUSAL, True),     # with softcap
    lowering.bwd_spec(torch.float16, 128, lowering.MASK_SLIDING, True),
]


@pytest.mark.parametrize("spec", SPECS, ids=lambda s: s.name()[:48])
def test_no_spills_and_no_early_reads_of_mfma_results(shim_built, spec):
    kernels = _kernels(spec)
    assert kernels
    for name, lines in kernels.items():
        if "delta" in name:
            continue
        assert any(ln.startswith("v_mfma") for ln in lines), name
        _check(name, lines)


def test_the_check_sees_an_early_read():
    lines = ["v_mfma_f32_32x32x16_bf16 a[0:15], v[0:3], v[4:7], a[0:15]", "v_add_u32_e32 v1, v2, v3",
             "v_accvgpr_read_b32 v9, a3"]
    with pytest.raises(AssertionError):
        _check("probe", lines)
    _check("probe", lines[:1] + ["s_nop 9", "s_nop 9"] + lines[1:])
    _check("probe", lines[:1] + ["v_mov_b32_e32 v0, v0"] * MIN_GAP + lines[2:])
    with pytest.raises(AssertionError):
        _check("probe", lines[:2] + ["scratch_load_dword v1, off, s0"])
    # a VGPR-destination MFMA of such a kernel: a copy of its accumulator before the drain is seen, one behind it is not
    chain = ["v_mfma_f32_32x32x16_bf16 a[0:15], v[0:3], v[4:7], a[0:15]",
             "v_mfma_f32_32x32x16_bf16 v[16:31], v[0:3], a[16:19], 0",
             "v_mfma_f32_32x32x16_bf16 v[16:31], v[4:7], a[20:23], v[16:31]"]
    with pytest.raises(AssertionError):
        _check("probe", chain + ["v_mov_b32_e32 v40, v17", "s_nop 9", "s_nop 9"])
    with pytest.raises(AssertionError):
        _check("probe", chain + ["global_load_dwordx4 v[28:31], v[0:1], off", "s_nop 9", "s_nop 9"])
    _check("probe", chain + ["v_add_u32_e32 v1, v2, v3", "s_nop 9", "s_nop 9", "v_mov_b32_e32 v40, v17"])


def _registers(operand):
    m = re.match(r"v\[(\d+):(\d+)\]$", operand) or re.match(r"v(\d+)$", operand)
    return set(range(int(m.group(1)), int(m.group(m.lastindex)) + 1)) if m else set()


def _check_settled(name, lines):
    """No MFMA reads a VGPR that the vector ALU wrote less than two wait states before: the compiler does not know that
    an inline MFMA needs them, for instance behind a copy of its own."""
    for i, ln in enumerate(lines):
        if not ln.startswith("v_mfma"):
            continue
        read = set().union(*(_registers(x.strip()) for x in ln.split(None, 1)[1].split(",")[1:]))
        states, j = 0, i - 1
        while j >= 0 and states < 2:
            x = lines[j]
            if x.startswith("v_") and not x.startswith("v_mfma"):
                dst = x.split(None, 1)[1].split(",")
                wrote = _registers(dst[0].strip()) | (_registers(dst[1].strip()) if "swap" in x else set())
                assert not wrote & read, f"{name}: '{ln}' reads what '{x}' wrote {states} wait states before"
            nop = re.match(r"s_nop (\d+)", x)
            states += int(nop.group(1)) + 1 if nop else 1
            j -= 1


@pytest.mark.parametrize("dtype,D,mask,softcap,blocks", [
    (torch.bfloat16, 128, lowering.MASK_CAUSAL, False, 2), (torch.float16, 128, lowering.MASK_NONE, False, 2),
    (torch.bfloat16, 128, lowering.MASK_CAUSAL, False, 1), (torch.float16, 128, lowering.MASK_SLIDING, True, 1),
    (torch.float16, 64, lowering.MASK_CAUSAL, False, 1)])
def test_hidden_accumulators_stay_in_their_registers(shim_built, dtype, D, mask, softcap, blocks):
    """lf_attn_bwd_dkdv hands its accumulators to the MFMAs as inputs: between the first and the last MFMA no other
    instruction may touch an AGPR, and nothing may be spilled."""
    lines = _kernels(lowering.bwd_spec(dtype, D, mask, softcap, key_blocks=blocks))["lf_attn_bwd_dkdv"]
    _check("lf_attn_bwd_dkdv", lines)
    _check_settled("lf_attn_bwd_dkdv", lines)
    mfma = [i for i, ln in enumerate(lines) if ln.startswith("v_mfma")]
    for ln in lines[mfma[0]:mfma[-1]]:
        assert ln.startswith("v_mfma") or not re.search(r"\ba(\d+|\[\d+:\d+\])", ln), ln
    # every accumulator tuple is written by MFMAs that name it as source and destination alike
    for ln in lines:
        m = re.match(r"v_mfma_\S+ (a\[\d+:\d+\]),.*, (\S+)$", ln)
        assert m is None or m.group(1) == m.group(2), ln


@pytest.mark.parametrize("threads", [256, 512])
@pytest.mark.parametrize("dtype,D,mask,softcap", [
    (torch.bfloat16, 128, lowering.MASK_CAUSAL, False), (torch.float16, 128, lowering.MASK_SLIDING, True),
    (torch.bfloat16, 128, lowering.MASK_NONE, True), (torch.float16, 64, lowering.MASK_SLIDING, False)])
def test_hidden_accumulators_of_dq_stay_in_their_registers(shim_built, dtype, D, mask, softcap, threads):
    lines = _kernels(lowering.bwd_spec(dtype, D, mask, softcap, dq_threads=threads))["lf_attn_bwd_dq"]
    _check("lf_attn_bwd_dq", lines)
    _check_settled("lf_attn_bwd_dq", lines)
    mfma = [i for i, ln in enumerate(lines) if ln.startswith("v_mfma")]
    for ln in lines[mfma[0]:mfma[-1]]:
        assert ln.startswith("v_mfma") or not re.search(r"\ba(\d+|\[\d+:\d+\])", ln), ln
    for ln in lines:
        m = re.match(r"v_mfma_\S+ (a\[\d+:\d+\]),.*, (\S+)$", ln)
        assert m is None or m.group(1) == m.group(2), ln


def _backward_builds():
    import __graft_entry__

    return sorted({s for s in __graft_entry__.standard_specs() if s.family == "bwd"}, key=lambda s: s.name())


@pytest.mark.parametrize("spec", _backward_builds(), ids=lambda s: s.name())
def test_every_backward_build_keeps_its_accumulators(shim_built, spec):
    """All checks of this file over every backward specialisation that the build compiles and a call can ask for."""
    kernels = _kernels(spec)
    for name in ("lf_attn_bwd_dkdv", "lf_attn_bwd_dq"):
        lines = kernels[name]
        _check(name, lines)
        _check_settled(name, lines)
        mfma = [i for i, ln in enumerate(lines) if ln.startswith("v_mfma")]
        for ln in lines[mfma[0]:mfma[-1]]:
            assert ln.startswith("v_mfma") or not re.search(r"\ba(\d+|\[\d+:\d+\])", ln), f"{name}: {ln}"
        for ln in lines:
            m = re.match(r"v_mfma_\S+ (a\[\d+:\d+\]),.*, (\S+)$", ln)
            assert m is None or m.group(1) == m.group(2), f"{name}: {ln}"


def test_every_split_the_rules_choose_is_built():
    """The rules for the work split -- key blocks, threads, queries split over the waves, dS kept where the rule says so and not
    where there is no room for it -- never leave the set of builds that the test above covers."""
    built, chosen = set(_backward_builds()), set()
    for dtype in (torch.bfloat16, torch.float16):
        for D in (64, 128):
            for mask in (lowering.MASK_NONE, lowering.MASK_CAUSAL, lowering.MASK_SLIDING):
                for cap in (False, True):
                    for units, group in ((1, 1), (1, 8), (31, 1), (50, 2), (100, 8), (256, 1), (4096, 4)):
                        for S in (1, 300, 1024, 2048, 8192):
                            q_split = lowering.bwd_q_split(D, mask, units, S)
                            blocks = units * group * lowering.bwd_ds_blocks(mask, 256, S, S)
                            for keep in {False, lowering.bwd_keep_ds(D, cap, units * group, group, S, blocks)}:
                                spec = lowering.bwd_spec(dtype, D, mask, cap, 1 if q_split else lowering.bwd_key_blocks(D, mask, cap, units, S),
                                                         lowering.bwd_dq_threads(D, mask, cap, units * group, S, S), keep, q_split,
                                                         lowering.bwd_grads_stay(2 * units * group * S * D))
                                assert spec in built, spec
                                chosen.add(spec)
    assert {("-DLF_BW_DS=1" in s.extra, "-DLF_BW_QSPLIT=1" in s.extra) for s in chosen} == {(a, b) for a in (False, True) for b in (False, True)}


def test_the_check_sees_an_unsettled_operand():
    mfma = "v_mfma_f32_32x32x16_bf16 v[16:31], v[0:3], v[4:7], v[16:31]"
    with pytest.raises(AssertionError):
        _check_settled("probe", ["v_mov_b32_e32 v17, v9", "v_add_u32_e32 v40, v1, v2", mfma])
    _check_settled("probe", ["v_mov_b32_e32 v17, v9", "s_nop 1", mfma])
    _check_settled("probe", ["v_mov_b32_e32 v32, v9", mfma])


@pytest.mark.parametrize("D,mask,softcap,window,kw", [
    (128, "sliding", 30.0, 64, {"key_blocks": 2}), (128, "sliding", None, 64, {"key_blocks": 2}),
    (128, "causal", 30.0, 0, {"key_blocks": 2}), (64, "causal", None, 0, {"key_blocks": 2}),
    (128, "causal", None, 0, {"key_blocks": 3}),
    (128, "causal", None, 0, {"dq_threads": 128})])
def test_backward_refuses_work_splits_that_no_kernel_is_built_for(D, mask, softcap, window, kw):
    """Two key blocks per wave are built and measured at head dim 128 without a window and a softcap only.  Anything else
    is refused before a kernel is built (the tensors here are not even on a GPU)."""
    q, k, v, o, dout = (torch.zeros((1, 2, 64, D), dtype=torch.bfloat16) for _ in range(5))
    plan = lowering.AttnPlan(mask=mask, window=window, scale=D ** -0.5, softcap=softcap)
    with pytest.raises(lowering.UnsupportedPlan, match=next(iter(kw))):
        lowering.attention_backward(q, k, v, o, torch.zeros((1, 2, 64)), dout, plan, **kw)


def test_backward_code_that_spills_is_refused(shim_built):
    """An accumulator that the compiler spills loses what the loop adds to it: ``compile_spec`` raises instead of handing
    out such code, here a build that reads twice as many fragments ahead as there are registers for."""
    spec = lowering.bwd_spec(torch.bfloat16, 128, lowering.MASK_SLIDING, True, key_blocks=2)
    spec = dataclasses.replace(spec, extra=spec.extra + ("-DLF_BW_PF=8",))
    with pytest.raises(RuntimeError, match="lf_attn_bwd_dkdv"):
        lowering.compile_spec(spec)
    code = lowering.compile_spec(lowering.bwd_spec(torch.bfloat16, 128, lowering.MASK_CAUSAL, key_blocks=2)).code_object
    assert runtime.private_segment_bytes(code) == {"lf_attn_bwd_delta": 0, "lf_attn_bwd_dkdv": 0, "lf_attn_bwd_dq": 0}
    with pytest.raises(ValueError):
        runtime.private_segment_bytes(b"no code object")


@pytest.mark.parametrize("bias,mask,softcap,paged,pack", [
    (b, m, c, pg, pk) for b in (1, lowering.MASK_BITS) for m, c, pg, pk in ((1, False, 3, 0), (2, False, 3, 0), (0, False, 0, 4), (2, True, 0, 4), (1, False, 3, 4))])
def test_masked_prefill_builds_and_does_not_spill(shim_built, bias, mask, softcap, paged, pack):
    """What the loop over dead tiles decides reaches the scalar operand of the direct loads (a decision left in a vector register
    does not assemble), and a branch around the products instead of that loop costs a second copy of O^T (spills)."""
    spec = lowering.KernelSpec("prefill_swp", 0, 128, mask, softcap, paged, 16 if paged else 1, bias=bias, pack=pack)
    assert not any("scratch_" in ln for ln in _kernels(spec)["lf_attn_prefill_swp"])


def test_boolean_masks_build_with_64_key_tiles_only(shim_built):
    with pytest.raises(RuntimeError, match="64-key tiles"):
        lowering.compile_spec(lowering.KernelSpec("prefill_swp", 0, 128, 0, False, bias=lowering.MASK_BITS, bn=32))


@pytest.mark.parametrize("spec,kernels", [
    (lowering.KernelSpec("prefill_swp", 0, 128, 1, False, bn=32), ["lf_attn_prefill_swp"]),
    (lowering.KernelSpec("prefill_swp", 1, 64, 0, False), ["lf_attn_prefill_swp"]),
    # (8 waves over 32-key tiles: the rows of a wave leave in two turns)
    (lowering.KernelSpec("prefill_swp", 0, 128, 0, False, bn=32, extra=("-DLF_NW=8", "-DLF_WPE=1")), ["lf_attn_prefill_swp"]),
    (lowering.bwd_spec(torch.bfloat16, 128, lowering.MASK_CAUSAL), ["lf_attn_bwd_dkdv", "lf_attn_bwd_dq"]),
    (lowering.bwd_spec(torch.float16, 64, lowering.MASK_SLIDING), ["lf_attn_bwd_dkdv", "lf_attn_bwd_dq"]),
], ids=["swp_bn32", "swp_d64", "swp_two_turns", "bwd_d128", "bwd_d64"])
def test_rows_that_meet_in_lds_are_written_before_they_are_read(spec, kernels, tmp_path):
    """The results' rows go from lane to lane through LDS without a barrier, a wave at a time.  Behind a kernel's last MFMA,
    writes and the reads on either side of them are kept apart by a wave barrier (a note to the compiler) or a workgroup's."""
    src, out = tmp_path / "kernel.hip", tmp_path / "kernel.s"
    src.write_text(spec.source())
    subprocess.run(["hipcc", "-x", "hip", "--offload-arch=gfx950", "--cuda-device-only", "-std=c++17", "-S", *spec.options(),
                    str(src), "-o", str(out)], check=True, capture_output=True)
    text = out.read_text()
    for name in kernels:
        body = text[text.index(f"\n{name}:"):text.index(f".size\t{name},")]
        tail = body[body.rindex("v_mfma"):]
        events = re.findall(r"ds_write|ds_read|wave barrier|s_barrier", tail)
        steps = [e for i, e in enumerate(events) if i == 0 or e != events[i - 1]]
        assert "ds_write" in steps and steps[-1] == "ds_read"
        for a, b in zip(steps, steps[1:]):
            assert {a, b} != {"ds_write", "ds_read"}, f"{name}: {steps}"
