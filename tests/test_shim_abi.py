"""The C-ABI library: loads, exports every symbol include/lf_shim.h declares, and its
host-side entry points (compile, cache, error reporting) behave.  No GPU, no launches."""
import ctypes
import os
import re

import pytest
import torch

from loopfuse_amd import lowering, runtime

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def header_symbols():
    text = open(os.path.join(ROOT, "include", "lf_shim.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(lf_[a-z0-9_]+)\s*\(", text)))


def test_exports_every_declared_symbol(shim_built):
    syms = header_symbols()
    assert len(syms) >= 13
    for s in syms:
        assert hasattr(shim_built, s), f"{s} declared in lf_shim.h but not exported"
    assert sorted(runtime.ABI_SYMBOLS) == syms
    assert shim_built.lf_abi_version() == 2


def test_compile_without_gpu_and_cache(shim_built, tmp_path):
    src = 'extern "C" __global__ void k(float* x) { x[threadIdx.x] *= 2.0f; }'
    code, hit, log = runtime.compile_source(src, "unit_k", ["-O3"], "gfx950", str(tmp_path))
    assert code[:4] == b"\x7fELF" and not hit
    code2, hit2, _ = runtime.compile_source(src, "unit_k", ["-O3"], "gfx950", str(tmp_path))
    assert hit2 and code2 == code
    # a different option is a different cache entry
    _, hit3, _ = runtime.compile_source(src, "unit_k", ["-O2"], "gfx950", str(tmp_path))
    assert not hit3
    assert len(os.listdir(tmp_path)) == 2


def test_compile_error_is_reported(shim_built):
    with pytest.raises(runtime.ShimError) as e:
        runtime.compile_source("this is not HIP", "bad", [], "gfx950", None)
    assert e.value.code != 0
    assert "error" in str(e.value).lower()


def test_bad_arguments_are_rejected(shim_built):
    L = shim_built
    assert L.lf_launch(None, 1, 1, 1, 64, 1, 1, 0, None, None) == -1
    assert b"null function" in L.lf_last_error()
    fn = ctypes.c_void_p()
    assert L.lf_get_function(ctypes.c_void_p(1234), b"k", ctypes.byref(fn)) == -1
    assert L.lf_module_unload(ctypes.c_void_p(1234)) == -1
    mod = ctypes.c_void_p()
    assert L.lf_module_load(None, 0, ctypes.byref(mod)) == -1


def test_launch_geometry_checks(shim_built):
    L = shim_built
    dummy = ctypes.c_void_p(1)
    assert L.lf_launch(dummy, 0, 1, 1, 64, 1, 1, 0, None, None) == -1
    assert L.lf_launch(dummy, 1, 1, 1, 2048, 1, 1, 0, None, None) == -1
    assert L.lf_launch(dummy, 1, 1, 1, 64, 1, 1, 200 * 1024, None, None) == -1


def test_params_struct_layout():
    from loopfuse_amd.lowering import AttnParams

    # 13 pointers, 26 int64 strides / spans, 12 ints, 3 floats (+4 bytes tail padding to the 8-byte alignment)
    assert AttnParams.q.offset == 0 and AttnParams.q2.offset == 88 and AttnParams.q_sb.offset == 104
    assert AttnParams.q2_sb.offset == 104 + 144
    assert AttnParams.k_span.offset == 104 + 192
    assert AttnParams.B.offset == 104 + 208
    assert AttnParams.k2_group.offset == 104 + 208 + 44
    assert AttnParams.scale.offset == 104 + 208 + 48
    assert AttnParams.denom_add.offset == 104 + 208 + 48 + 8
    assert ctypes.sizeof(AttnParams) == 376


@pytest.mark.parametrize("host,mirror,device,source", [
    ("LfAttnParamsHost", "AttnParams", "LfAttnParams", "lf_common.hip.h"),
    ("LfAttnBwdParamsHost", "AttnBwdParams", "LfAttnBwdParams", "lf_attn_bwd.hip"),
])
def test_c_header_matches_the_ctypes_mirror_and_the_device_struct(tmp_path, host, mirror, device, source):
    """include/lf_attn_params.h (C hosts), the ctypes structure of lowering.py and the device
    struct list the same fields at the same offsets."""
    import subprocess

    from loopfuse_amd import lowering

    mirror = getattr(lowering, mirror)
    names = [n for n, _ in mirror._fields_]
    prog = "#include <stdio.h>\n#include <stddef.h>\n#include \"lf_attn_params.h\"\nint main(void) {\n"
    for n in names:
        prog += f'  printf("{n} %zu\\n", offsetof({host}, {n}));\n'
    prog += f'  printf("sizeof %zu\\n", sizeof({host}));\n  return 0;\n}}\n'
    src = tmp_path / "off.c"
    src.write_text(prog)
    exe = tmp_path / "off"
    subprocess.run(["gcc", "-std=c11", "-I" + os.path.join(ROOT, "include"), str(src), "-o", str(exe)], check=True)
    out = dict(line.split() for line in subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.splitlines())
    for n in names:
        assert int(out[n]) == getattr(mirror, n).offset, n
    assert int(out["sizeof"]) == ctypes.sizeof(mirror)
    # the device struct declares the same field names in the same order
    dev = open(os.path.join(ROOT, "loopfuse_amd", "csrc", "kernels", source)).read()
    body = dev[dev.index("struct %s {" % device):]
    body = re.sub(r"//[^\n]*", "", body[:body.index("};")])
    fields = []
    for decl in body.split("{", 1)[1].split(";"):
        decl = decl.strip()
        if decl:
            fields += [re.sub(r"[^A-Za-z0-9_]", "", x.split()[-1]) for x in decl.split(",")]
    assert fields == names


def _stubbed_static_step(monkeypatch, B, Hq, Hkv, S, page, D=128):
    """``attention(..., static_scratch=True)`` on the CPU with the launch replaced by the library's own size check;
    returns the number of splits."""
    room, seen = runtime.static_scratch_bytes(), []

    def launch(decode, combine, P, acc, ml, grid, *rest):
        if (acc + 255) // 256 * 256 + (ml + 255) // 256 * 256 > room:
            raise runtime.ShimError("static", -4, "too large")
        seen.append((P.nsplit, P.split_len, grid[1]))

    monkeypatch.setattr(lowering, "_check_tensor", lambda *a: None)
    monkeypatch.setattr(lowering, "get_kernel", lambda *a: None)
    monkeypatch.setattr(runtime, "launch_decode_static", launch)
    q = torch.empty((B, Hq, 1, D), dtype=torch.bfloat16)
    pool = torch.empty((1, page, Hkv, D) if page > 1 else (1, Hkv, D), dtype=torch.bfloat16)
    pool = pool.expand(B * S // page, *pool.shape[1:])

    class Table(torch.Tensor):
        is_cuda = True

    table = torch.zeros((B, S // page), dtype=torch.int32).as_subclass(Table)
    plan = lowering.AttnPlan(scale=D ** -0.5, k_paged=True, v_paged=True)
    lowering.attention(q, pool, pool, plan, table, table, out=torch.empty_like(q), static_scratch=True)
    (nsplit, split_len, gy), = seen
    assert nsplit == gy == -(-S // split_len)
    return nsplit


# what decode_split made of these with the per-wave loads: two splits, or as many as have room
@pytest.mark.parametrize("B,Hq,Hkv,S,page", [(96, 16, 16, 1024, 16), (112, 16, 16, 8192, 64), (180, 8, 8, 1024, 16), (224, 8, 8, 8192, 16),
                                             (16, 64, 8, 8192, 1), (16, 32, 4, 8192, 1), (4, 64, 8, 8192, 2)])
def test_static_scratch_serves_what_the_general_split_rule_fits(shim_built, monkeypatch, B, Hq, Hkv, S, page):
    splits = _stubbed_static_step(monkeypatch, B, Hq, Hkv, S, page)
    assert splits >= 2 and 4 * B * Hq * splits * 130 <= runtime.static_scratch_bytes()


def test_static_scratch_split_rule():
    """Over sizes: a step runs wherever one of the two rules' counts does, with the cooperative rule's if that one runs."""
    room, D = 8 << 20, 128
    upto = lambda n: -(-n // 256) * 256
    for rows in (1, 8, 100, 1000, 2000, 4096, 10000):
        for Sk in (64, 1000, 1024, 2048, 8192, 32768):
            runs = lambda n: (k := lowering._split_lengths(n, Sk)[0]) > 1 and upto(4 * rows * k * D) + upto(8 * rows * k) <= room
            for n in (1, 2, 5, 16, 33, 64):
                for plain in (1, 2, 4, 16, 64):
                    got = lowering.decode_static_split(n, plain, Sk, rows, D, room)
                    assert runs(got) if runs(plain) or runs(n) else got == n or (1 < got < n and runs(got))
                    assert got == n or not runs(n)
    assert lowering.decode_static_split(16, 4, 8192, 1024, D, room) == 15


def test_switches_are_read_from_the_environment_of_the_moment(monkeypatch):
    """Set, unset, and with ``os.environ`` itself replaced by another mapping."""
    assert lowering.decode_split(1, 1 << 16) == 64
    monkeypatch.setenv("LOOPFUSE_DECODE_SPLITS", "5")
    assert lowering.decode_split(1, 1 << 16) == 5
    monkeypatch.delenv("LOOPFUSE_DECODE_SPLITS")
    assert lowering.decode_split(1, 1 << 16) == 64
    monkeypatch.setattr(os, "environ", {"LOOPFUSE_DECODE_SPLITS": "3"})
    assert lowering.decode_split(1, 1 << 16) == 3


def test_a_captured_call_keeps_no_scratch_that_a_later_call_lets_go_of(monkeypatch):
    """Under graph capture the split-K scratch is neither taken from nor put into the buffer that calls on a stream share:
    that one is replaced, and its memory given back, as soon as a larger one is needed, and the graph goes on writing to it."""
    monkeypatch.setattr(lowering, "_scratch", {})
    monkeypatch.setattr(runtime, "current_stream_handle", lambda: 7)
    capturing = [False]
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing[0])
    dev = torch.device("cpu")
    shared = lowering._get_scratch(dev, 10)
    assert lowering._get_scratch(dev, 1 << 20) is shared
    capturing[0] = True
    own = lowering._get_scratch(dev, 1 << 22)
    assert own.numel() == 1 << 22 and own.data_ptr() != shared.data_ptr()
    assert list(lowering._scratch.values()) == [shared]
    assert lowering._get_scratch(dev, 10).data_ptr() != shared.data_ptr()


@pytest.mark.parametrize("units,Sk,page,pays", [
    (64, 2048, 1, True), (64, 2048, 16, True), (28, 4096, 16, True),      # whole rounds of even splits
    (264, 228, 1, False), (276, 2192, 16, False), (285, 1728, 16, False),  # a second round of a few workgroups
    (8, 1200, 4, False), (16, 2048, 16, False), (250, 2048, 16, True)])    # too few workgroups; almost a round
def test_cooperative_decode_is_chosen_where_its_rounds_are_full(units, Sk, page, pays):
    assert lowering.decode_coop_pays(units, Sk, 1, page) == pays


@pytest.mark.parametrize("units,Sk,rows", [(64, 2048, 8), (66, 871, 8), (50, 1142, 8), (8, 8192, 4), (300, 100, 1), (1, 32768, 16)])
def test_cooperative_split_count(units, Sk, rows):
    """Within its bounds, and of the counts it looks at the one with the least cost."""
    n = lowering.decode_coop_split(units, Sk, rows)
    most = max(1, min(64, Sk // 160))
    assert 1 <= n <= most
    for m in (1, 256 // units, 512 // units):
        m = max(1, min(most, m))
        assert lowering._coop_cost(n, units, Sk, rows) <= lowering._coop_cost(m, units, Sk, rows)


@pytest.mark.parametrize("workgroups,keys,tile", [(767, 100, 0), (768, 2047, 32), (768, 2048, 0), (2047, 8192, 0), (2048, 8192, 32)])
def test_kv_tile_rule(workgroups, keys, tile):
    assert lowering.prefill_kv_tile(128, workgroups=workgroups, keys=keys) == tile
    assert lowering.prefill_kv_tile(64, workgroups=workgroups, keys=keys) == 0


def test_a_split_step_and_its_merge_are_launched_together(shim_built, monkeypatch):
    """Threads that decode on one stream share its scratch: no step of another thread comes between a step and its merge."""
    import threading
    import time

    order = []

    class Fake:
        def __init__(self, name):
            self.name = name

        def launch(self, *args):
            order.append((threading.get_ident(), self.name))
            time.sleep(0.002)

    monkeypatch.setattr(lowering, "_check_tensor", lambda *a: None)
    monkeypatch.setattr(lowering, "_kernels_of", lambda spec: {n: Fake(n) for n in ("lf_attn_decode", "lf_attn_decode_combine")})
    monkeypatch.setattr(lowering, "_scratch", {})
    monkeypatch.setattr(runtime, "current_stream_handle", lambda: 0)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    q, k = torch.zeros((1, 2, 1, 64), dtype=torch.bfloat16), torch.zeros((1, 2, 256, 64), dtype=torch.bfloat16)

    def work():
        for _ in range(5):
            lowering.attention(q, k, k, lowering.AttnPlan(scale=0.125), num_splits=2)

    threads = [threading.Thread(target=work) for _ in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(order) == 30
    for (a, first), (b, second) in zip(order[::2], order[1::2]):
        assert (a, first, second) == (b, "lf_attn_decode", "lf_attn_decode_combine")
