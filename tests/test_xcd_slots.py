"""Workgroup -> (unit, tile) mapping of the prefill and backward kernels (``lf_slot_of_block``).

CPU: the device function itself, compiled as host C++, covers every (unit, tile) exactly once over the grid
``lowering.xcd_slots`` asks for, longest tiles first inside a group.  GPU: forward and backward at numbers of
(batch, head) units that are cut into parts (1, 3, 9, 12) against float64."""
import ctypes
import os
import subprocess

import pytest
import torch

from loopfuse_amd import lowering, runtime


@pytest.fixture(scope="module")
def slot_of_block(tmp_path_factory):
    text = open(os.path.join(runtime.KERNEL_DIR, "lf_prefill_blocks.hip.h")).read()
    a = text.index("__device__ __forceinline__ bool lf_slot_of_block")
    body = text[a:text.index("\n}\n", a) + 3].replace("__device__ __forceinline__", "static")
    d = tmp_path_factory.mktemp("slots")
    src, out = d / "slots.cpp", d / "slots.so"
    src.write_text("#include <algorithm>\nusing std::min;\n" + body +
                   'extern "C" int slot(unsigned b, int u, int t, int g, int* unit, int* tile) '
                   "{ return lf_slot_of_block(b, u, t, g, *unit, *tile); }\n")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wno-unknown-pragmas", "-shared", "-fPIC", str(src), "-o", str(out)], check=True)
    return ctypes.CDLL(str(out)).slot


@pytest.mark.parametrize("group", [4, 8])
@pytest.mark.parametrize("units", [1, 2, 3, 7, 8, 9, 12, 31, 64, 65, 100, 257])
@pytest.mark.parametrize("tiles", [1, 2, 5, 8, 47, 64])
def test_every_tile_once(slot_of_block, units, tiles, group):
    grid = lowering.xcd_slots(units, tiles)
    # a host that still launches the padded grid of whole groups starts at least as many workgroups
    assert grid <= 8 * (((units + 7) // 8 + group - 1) // group * group) * tiles
    seen, per_xcd = {}, [0] * 8
    unit, tile = ctypes.c_int(), ctypes.c_int()
    for b in range(grid + 16):
        if slot_of_block(b, units, tiles, group, ctypes.byref(unit), ctypes.byref(tile)):
            key = (unit.value, tile.value)
            assert key not in seen and 0 <= key[0] < units and 0 <= key[1] < tiles
            seen[key] = b
            per_xcd[b % 8] += 1
    assert len(seen) == units * tiles
    assert grid == 8 * (max(seen.values()) // 8 + 1)                   # no slot row of the grid is padding alone
    if units * tiles >= 64 and tiles >= 8:
        assert max(per_xcd) <= 1.125 * units * tiles / 8 + 1           # no XCD carries much more than its share
    for u in range(units):                                             # dispatch order: a unit's tiles in order per part
        order = [seen[(u, t)] for t in range(tiles)]
        assert all(order[t] < order[t + 8] for t in range(tiles - 8))


@pytest.mark.gpu
@pytest.mark.parametrize("B,Hq,Hkv,S,D,mask,window", [(1, 1, 1, 700, 128, "causal", 0), (1, 4, 1, 333, 128, "causal", 0),
                                                      (3, 6, 3, 260, 64, "sliding", 70), (1, 12, 12, 129, 64, None, 0)])
def test_cut_units_forward_and_backward(B, Hq, Hkv, S, D, mask, window):
    from test_backward_gpu import _ref
    g = torch.Generator().manual_seed(S)
    q, k, v, dout = (torch.randn(s, generator=g).bfloat16().cuda() for s in ((B, Hq, S, D), (B, Hkv, S, D), (B, Hkv, S, D), (B, Hq, S, D)))
    plan = lowering.AttnPlan(mask=mask, window=window, scale=D ** -0.5)
    lse = torch.empty((B, Hq, S), dtype=torch.float32, device="cuda")
    o = lowering.attention(q, k, v, plan, lse=lse)
    got = (o, *lowering.attention_backward(q, k, v, o, lse, dout, plan))
    want = _ref(q, k, v, dout, mask, window, D ** -0.5)
    # bf16 inputs, probabilities and results: 2^-9 relative rounding each, a few of them per value
    for a, w in zip(got, (want[0], *want[2:])):
        assert ((a.double() - w).norm() / w.norm()).item() <= 1e-2
    # the register-staged kernel walks pairs of q tiles through the same mapping
    o2 = lowering.attention(q, k, v, plan, force_family="prefill", choice={"prefill": "w32"})
    assert ((o2.double() - want[0]).norm() / want[0].norm()).item() <= 1e-2
