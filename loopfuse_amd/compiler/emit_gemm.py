"""MFMA lowering of a contraction nest with its pointwise epilogue fused -- the counterpart of the
``tl.dot`` the reference emits for every contraction (``loopfuse/codegen.py:658-668``; its accuracy
cases ``tests/test_accuracy.py:56-82``: ``a @ b + c`` in two and three dims).

A nest ``out[batch.., m, n] = f(sum_k A[batch.., m, k] * B[batch.., k, n], other reads)`` with bf16 /
fp16 operands becomes one kernel.  A workgroup owns a tile of the output -- 64 x 128 to 256 x 256,
four or eight waves (``TILES``), a compile-time choice -- and walks k, or a part of it, in
steps of 64.  Both operand tiles arrive by direct global -> LDS loads
(``buffer_load_dwordx4 ... lds``: 16-byte pieces, range-checked so that the edges arrive as zeros, the XOR
permutation applied on the global side), two to four stages, one barrier per step, and come back as
``v_mfma_f32_32x32x16`` operands -- by plain 16-byte reads where k is the contiguous dimension of the
operand in memory, by transposed reads (``ds_read_b64_tr_b16``) where m / n is.  The product is formed
transposed (C^T = B^T A^T); the fp32 accumulators then pass through LDS once so that a lane holds four
consecutive n of one m and neighbouring lanes neighbouring n: the epilogue expression -- whatever the
fused nest holds around the contraction -- is evaluated there per element, its reads coalesced, and the
results leave in 8- or 16-byte stores along the rows of the output.  Where the tiles alone would leave
CUs idle, k is split into parts (``choose``): the workgroups then leave fp32 partial sums, which a second
kernel adds up and runs the epilogue on.  Tiles are walked in bands of a few
tile rows, an XCD taking a contiguous run of them, so that its resident workgroups share operand rows and
columns in its L2.

Which of the two layouts an operand has is a compile-time flag of the kernel (``-DLFG_A_ROWS``,
``-DLFG_B_ROWS``); the launcher picks the code object per call from the strides.  Calls the kernel
cannot serve (strides that are not multiples of 8 elements, k or the contiguous extent not a multiple
of 8, unaligned bases, an operand beyond the 32-bit byte offsets of the loads) take the plain
one-thread-per-element kernel of the same nest.
"""
from __future__ import annotations

import dataclasses
import functools
import math
from typing import Optional

from . import ir
from .emit import _CT, MAX_N, MAX_PTR, Emitter, Kernel, NotLowerable

BK = 64
# Workgroup tiles: waves along m, waves along n, 32 x 32 blocks per wave along m, along n, LDS stages.  128 x 128 on four
# waves at two workgroups per CU (s), or on eight with four stages, one per CU (d: a step does not cost a memory latency where
# there are too few tiles for two); 256 x 128 on eight waves (m) and 256 x 256 (l), one per CU, with three quarters and half
# the L2 -> LDS bytes per flop; 64 x 128 on four (n), up to two per CU, for few rows of A, where the tiles' number, not their
# bytes, is the time.
TILES = {"s": (2, 2, 2, 2, 2), "d": (4, 2, 1, 2, 4), "m": (4, 2, 2, 2, 3), "l": (4, 2, 2, 4, 2), "n": (2, 2, 1, 2, 3)}


def tile_extent(shape: str) -> tuple:
    wm, wn, mb, nb, _ = TILES[shape]
    return 32 * wm * mb, 32 * wn * nb


def tile_options(shape: str, split: bool = False, b_streams: bool = False) -> list:
    wm, wn, mb, nb, stages = TILES[shape]
    return [f"-DLFG_WGM={wm}", f"-DLFG_WGN={wn}", f"-DLFG_MB={mb}", f"-DLFG_NB={nb}", f"-DLFG_STAGES={stages}"] + \
        (["-DLFG_SPLIT=1"] if split else []) + (["-DLFG_B_NT=1"] if b_streams else [])

GEMM_PRELUDE = r"""
typedef float lfg_f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned int lfg_u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int lfg_u32x2 __attribute__((ext_vector_type(2)));
typedef float lfg_f32x4 __attribute__((ext_vector_type(4)));
typedef short lfg_s16x4 __attribute__((ext_vector_type(4)));
#ifndef LFG_SPLIT
#define LFG_SPLIT 0      /* 1: a workgroup sums a part of k and leaves fp32 partials; a second kernel adds them up and runs the epilogue */
#endif
#ifndef LFG_B_NT
#define LFG_B_NT 0       /* 1: B by non-temporal loads */
#endif
typedef __bf16 lfg_bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 lfg_f16x8 __attribute__((ext_vector_type(8)));
__device__ __forceinline__ lfg_f32x16 lfg_mfma(__bf16, lfg_u32x4 a, lfg_u32x4 b, lfg_f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(lfg_bf16x8, a), __builtin_bit_cast(lfg_bf16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ lfg_f32x16 lfg_mfma(_Float16, lfg_u32x4 a, lfg_u32x4 b, lfg_f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(lfg_f16x8, a), __builtin_bit_cast(lfg_f16x8, b), c, 0, 0, 0);
}
// Operand tiles in LDS; `kExtent` = rows / columns of the workgroup's tile along m (A) or n (B), 64 k per step.
//   k-contiguous operand ("rows"): [kExtent rows][64 k]; the eight 16-byte pieces of a row are permuted by the
//   row pair, so that the 16-byte reads of 16 consecutive rows touch every bank once.
//   m/n-contiguous operand ("cols"): [64 k][kExtent]; the 64-byte groups of a row are permuted by the row, for the
//   transposed reads (4 consecutive rows x 64 contiguous bytes per 32 lanes); of 64 columns two rows share the banks' span.
__device__ __forceinline__ int lfg_rows_at(int row, int piece) { return row * 64 + 8 * (piece ^ ((row >> 1) & 7)); }
template <int kExtent>
__device__ __forceinline__ int lfg_cols_swz(int row) { return kExtent >= 128 ? 4 * (row & 3) : 4 * ((row >> 1) & 1); }
template <int kExtent>
__device__ __forceinline__ int lfg_cols_at(int row, int piece) { return row * kExtent + 8 * (piece ^ lfg_cols_swz<kExtent>(row)); }
// Tiles arrive by direct global -> LDS loads: a wave-level load writes 64 lanes x 16 bytes at M0 + 16 * lane, i.e. 64
// consecutive 16-byte positions `idx` of the tile, and the permutation is applied on the global side: the lane that
// fills position idx fetches the piece (outer = m or n, k) that lives there.
template <bool kRows, int kExtent> struct LfgPiece {
  static __device__ __forceinline__ int outer(int idx) {
    return kRows ? (idx >> 3) : 8 * ((idx % (kExtent / 8)) ^ lfg_cols_swz<kExtent>(idx / (kExtent / 8)));
  }
  static __device__ __forceinline__ int k(int idx) {
    return kRows ? 8 * ((idx & 7) ^ ((idx >> 4) & 7)) : idx / (kExtent / 8);
  }
};
// Buffer resource over `bytes` bytes from `base` (raw buffer, 32-bit offsets, range checked: a load beyond the range
// delivers zeros)
__device__ __forceinline__ lfg_u32x4 lfg_make_buffer(const void* base, unsigned bytes) {
  const unsigned long long a = (unsigned long long)base;
  lfg_u32x4 rs;
  rs[0] = __builtin_amdgcn_readfirstlane((unsigned)a);
  rs[1] = __builtin_amdgcn_readfirstlane((unsigned)(a >> 32) & 0xffffu);
  rs[2] = __builtin_amdgcn_readfirstlane(bytes);
  rs[3] = 0x00020000u;
  return rs;
}
// One wave-level direct-to-LDS load (not tracked by the compiler's wait counters: callers wait with s_waitcnt vmcnt);
// kNt: non-temporal, for an operand that is not read again
template <bool kNt>
__device__ __forceinline__ void lfg_dma(const lfg_u32x4& rs, unsigned voff, unsigned lds_addr) {
  unsigned m0_written;
  if (kNt)
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %3, 0 offen nt lds"
                 : "={m0}"(m0_written) : "s"(lds_addr), "v"(voff), "s"(rs) : "memory");
  else
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %3, 0 offen lds"
                 : "={m0}"(m0_written) : "s"(lds_addr), "v"(voff), "s"(rs) : "memory");
}
// This wave's loads but the newest `n` have landed and its LDS reads are done; then the workgroup's barrier.  The wait is
// the builtin, so that the compiler knows its own reads to be done and does not wait for them again.
#define LFG_STAGE_BARRIER(n)                                                         \
  do {                                                                               \
    asm volatile("" ::: "memory");                                                   \
    __builtin_amdgcn_s_waitcnt(((n) & 15) | 0x70 | (((n) >> 4) << 14));              \
    __builtin_amdgcn_s_barrier();                                                    \
    asm volatile("" ::: "memory");                                                   \
  } while (0)
// MFMA operand (either side: 32 rows or columns `blk`, lane % 32 picks one, lane / 32 the half of the 16-step `ks`):
// k = 16 * ks + 8 * (lane / 32) .. + 7 in both layouts
template <bool kRows, int kExtent>
__device__ __forceinline__ lfg_u32x4 lfg_operand(const unsigned short* tile, int blk, int ks, int lane) {
  const int l32 = lane & 31, g = lane >> 5;
  if (kRows) return *reinterpret_cast<const lfg_u32x4*>(&tile[lfg_rows_at(32 * blk + l32, 2 * ks + g)]);
  const int j16 = lane & 15, dh = (lane >> 4) & 1;
  const int col = 32 * blk + 16 * dh + 4 * (j16 & 3);
  lfg_u32x2 h[2];
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    const int row = 16 * ks + 8 * g + 4 * half + (j16 >> 2);
    const unsigned short* src = &tile[lfg_cols_at<kExtent>(row, col >> 3) + (col & 7)];
    const lfg_s16x4 t = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) lfg_s16x4*)(src));
    h[half] = __builtin_bit_cast(lfg_u32x2, t);
  }
  return lfg_u32x4{h[0][0], h[0][1], h[1][0], h[1][1]};
}
// four consecutive results of one output row: one store when the row is contiguous and aligned, else element-wise
template <typename T> struct LfgPack;
template <> struct LfgPack<float> { typedef lfg_u32x4 type; };
template <> struct LfgPack<__bf16> { typedef lfg_u32x2 type; };
template <> struct LfgPack<_Float16> { typedef lfg_u32x2 type; };
template <typename T>
__device__ __forceinline__ void lfg_st4(void* p, long long at, const float (&r)[4]) {
  T t[4] = {(T)r[0], (T)r[1], (T)r[2], (T)r[3]};
  typedef typename LfgPack<T>::type pack_t;
  *reinterpret_cast<pack_t*>(reinterpret_cast<T*>(p) + at) = __builtin_bit_cast(pack_t, t);
}
"""


@dataclasses.dataclass
class GemmInfo:
    """What the launcher needs besides the usual parameter block."""
    m: ir.Atom
    n: ir.Atom
    k: ir.Atom
    batch: list                 # parallel atoms other than m, n (outer to inner)
    a_buf: ir.Buffer
    b_buf: ir.Buffer
    a_dims: tuple               # (dim of A indexed by m, dim indexed by k)
    b_dims: tuple               # (dim of B indexed by n, dim indexed by k)
    a_batch_dims: list          # dims of A indexed by a batch atom
    b_batch_dims: list
    b_batch: list               # the batch atoms that index them
    flags_at: int = 0           # n[flags_at]: the output's rows are contiguous and aligned for 8- / 16-byte stores;
                                # n[flags_at + 1], n[flags_at + 2]: bytes of A / B reachable from a batch element's base;
                                # n[flags_at + 3], n[flags_at + 4]: parts that k is split into, steps of 64 k per part
    out_buf: object = None
    out_n_dim: int = -1         # dimension of the output indexed by n alone (-1: none)
    ws_ptr: int = 0             # ptr[ws_ptr]: fp32 partials of a split product
    sum_source: str = ""        # the kernel that adds them up


def _single(atoms) -> Optional[ir.Atom]:
    """The one atom of extent > 1 that indexes a buffer dimension; None for a dimension of extent 1."""
    xs = [a for a in ir.leaves(atoms) if a.hint != 1]
    if len(xs) > 1 or any(a.broadcast for a in xs):
        raise NotLowerable("an operand dimension indexed by several atoms")
    return xs[0] if xs else None


def match(nest: ir.Nest, dtypes: dict) -> Optional[GemmInfo]:
    """The nest as batched matrix product + pointwise epilogue, or None."""
    s = nest.stmt
    if not isinstance(s, ir.Assign) or [a for a in ir.leaves(nest.red) if a.hint != 1]:
        return None
    dots = [e for e in ir.walk(s.value) if isinstance(e, ir.Dot)]
    if len(dots) != 1:
        return None
    d = dots[0]
    if not (isinstance(d.a, ir.Read) and isinstance(d.b, ir.Read)) or d.a.gather is not None or d.b.gather is not None:
        return None
    if dtypes.get(d.a.buf.name) not in (1, 2) or dtypes.get(d.a.buf.name) != dtypes.get(d.b.buf.name):
        return None
    over = [a for a in ir.leaves(d.over) if a.hint != 1]
    par = [a for a in ir.leaves(nest.par) if a.hint != 1]
    if len(over) != 1:
        return None
    k = over[0]
    try:
        ia = [_single(x) for x in d.a.idx]
        ib = [_single(x) for x in d.b.idx]
    except NotLowerable:
        return None

    def has(lst, a):
        return any(x is a for x in lst)

    ms = [a for a in par if has(ia, a) and not has(ib, a)]
    ns = [a for a in par if has(ib, a) and not has(ia, a)]
    if not ms or not ns or not has(ia, k) or not has(ib, k):
        return None
    m, n = ms[-1], ns[-1]          # the innermost one of each side; outer ones (a view of [.., M, K] rows) count as batch
    batch = [a for a in par if a is not m and a is not n]
    if any(x is not None and x is not m and x is not k and not has(batch, x) for x in ia) or \
            any(x is not None and x is not n and x is not k and not has(batch, x) for x in ib):
        return None
    # each of m, n, k indexes exactly one dimension of its operand
    if sum(x is m for x in ia) != 1 or sum(x is k for x in ia) != 1 or sum(x is n for x in ib) != 1 or sum(x is k for x in ib) != 1:
        return None
    pos = lambda lst, a: next(i for i, x in enumerate(lst) if x is a)      # noqa: E731
    return GemmInfo(m, n, k, batch, d.a.buf, d.b.buf, (pos(ia, m), pos(ia, k)), (pos(ib, n), pos(ib, k)),
                    [i for i, x in enumerate(ia) if x is not None and has(batch, x)],
                    [i for i, x in enumerate(ib) if x is not None and has(batch, x)],
                    [x for x in ib if x is not None and has(batch, x)])


def b_batches(info: GemmInfo, ext: dict, stride) -> tuple:
    """(matrices B that the batch holds, batch elements that share each): an atom shares B where it does not index it or, in an
    expanded tensor, does not move along it (``stride(d)`` of its dimension d)."""
    own = [a for d, a in zip(info.b_batch_dims, info.b_batch) if stride(d)]
    return math.prod(ext[a.id] for a in own), math.prod(ext[a.id] for a in info.batch if not any(a is x for x in own))


class GemmEmitter(Emitter):
    """HIP source of a contraction nest on the MFMA path."""

    def __init__(self, nest: ir.Nest, dtypes: dict, name: str, info: GemmInfo):
        super().__init__(nest, dtypes, name)
        self.info = info
        self.reads: list = []       # what the epilogue reads besides the product, loaded ahead of it (rd[k])
        self.conditional = 0

    def expr(self, e: ir.Expr) -> str:
        if isinstance(e, ir.Dot):
            return "accv"
        if isinstance(e, ir.Select):
            self.conditional += 1
            try:
                return super().expr(e)
            finally:
                self.conditional -= 1
        if isinstance(e, ir.Read) and e.gather is None and not self.conditional:
            self.reads.append(super().expr(e))
            return f"rd[{len(self.reads) - 1}]"
        return super().expr(e)

    def emit(self) -> Kernel:
        g, n = self.info, self.nest
        par = [a for a in ir.leaves(n.par) if a.hint != 1]
        for a in par:
            self.atom(a)
        km, kn, kk = self.atom(g.m), self.atom(g.n), self.atom(g.k)
        ia, ib = self.buf(g.a_buf), self.buf(g.b_buf)
        elem = _CT[self.dtypes[g.a_buf.name]]

        def base(buf, ptr, read_idx, batch_dims):
            terms = []
            for d in batch_dims:
                a = _single(read_idx[d])
                terms.append(f"i{self.atom(a)} * S{self.stride(buf, d)}")
            return f"reinterpret_cast<const {elem}*>(p.ptr[{ptr}]) + ({' + '.join(terms) or '0ll'})"

        dot = next(e for e in ir.walk(n.stmt.value) if isinstance(e, ir.Dot))
        a_base = base(g.a_buf, ia, dot.a.idx, g.a_batch_dims)
        b_base = base(g.b_buf, ib, dot.b.idx, g.b_batch_dims)
        sam, sak = self.stride(g.a_buf, g.a_dims[0]), self.stride(g.a_buf, g.a_dims[1])
        sbn, sbk = self.stride(g.b_buf, g.b_dims[0]), self.stride(g.b_buf, g.b_dims[1])
        val = self.expr(n.stmt.value)              # epilogue on `accv`; registers its buffers, strides, scalars
        if self.lines:
            raise NotLowerable("a second contraction inside the epilogue")
        # The reads of all elements go out before the first of them is needed: an activation with branches (erf) keeps the
        # compiler from moving the loads of the next element above it, which then waits for memory once per element.  With
        # the sum's block numbers divided in 32 bits, linear -> gelu -> linear with 256 rows, 4096 / 16384 wide: 106.4 -> 104.9
        # us, 1024 rows 287.9 -> 282.4, 64 rows 65.0 -> 64.0.  (Two blocks of columns per workgroup of the sum: no more at 256
        # and 1024 rows, 64 rows 64.9 -> 66.1: half the workgroups.)
        lambdas = f"""constexpr int kRd = {max(1, len(self.reads))};
  auto read = [&](float* rd, long long i{km}, long long i{kn}) {{ {' '.join(f'rd[{j}] = {r};' for j, r in enumerate(self.reads))} }};
  auto epilogue = [&](float accv, const float* rd, long long i{km}, long long i{kn}) -> float {{ return {val}; }};"""
        out = n.writes()
        o = self.buf(out)
        ooff = self.offset(out, out.dims, None)
        g.out_buf = out
        for d, atoms in enumerate(out.dims):
            xs = [a for a in ir.leaves(atoms) if a.hint != 1]
            if len(xs) == 1 and xs[0] is g.n:
                g.out_n_dim = d
        na, ns = len(self.atoms), len(self.strides)
        g.flags_at = na + ns
        g.ws_ptr = len(self.bufs)
        if na + ns + 5 > MAX_N or len(self.bufs) + 1 > MAX_PTR:
            raise NotLowerable("nest touches too many buffers / dimensions")
        defs = [f"const long long N{k} = p.n[{k}];" for k in range(na)] + \
               [f"const long long S{k} = p.n[{na + k}];" for k in range(ns)]
        batch_decode = []
        for a in reversed(g.batch):
            k = self.atom(a)
            batch_decode.append(f"const long long i{k} = blk % N{k}; blk /= N{k};")
        out_t = _CT[self.dtypes[out.name]]
        src = f"""extern "C" __global__ void __launch_bounds__(64 * LFG_WGM * LFG_WGN, 2)
{self.name}(const LfGenParams p) {{
  {' '.join(defs)}
  constexpr bool a_rows = LFG_A_ROWS != 0, b_rows = LFG_B_ROWS != 0;
  // the workgroup's tile: kWM x kWN waves, each kMB x kNB blocks of 32 x 32
  constexpr int kWM = LFG_WGM, kWN = LFG_WGN, kMB = LFG_MB, kNB = LFG_NB;
  constexpr int kBM = 32 * kWM * kMB, kBN = 32 * kWN * kNB, kWaves = kWM * kWN, kNT = 64 * kWaves;
  constexpr int kTileA = kBM * {BK}, kTileB = kBN * {BK};                    // elements of one operand tile
  constexpr int kPA = kBM * 8 / kNT, kPB = kBN * 8 / kNT;                   // 16-byte pieces per thread and tile
  constexpr int kS = LFG_STAGES;
  static_assert(kNB % 2 == 0 && kBM * 8 % kNT == 0 && kBN * 8 % kNT == 0, "tile shape");
  static_assert(LFG_SPLIT || kWaves * kMB * 8192 <= 2 * kS * (kTileA + kTileB), "the accumulators pass through the tiles' LDS");
  static_assert((kS - 1) * (kPA + kPB) < 64, "loads in flight behind a stage");
  __shared__ __attribute__((aligned(16))) unsigned short lds[kS * (kTileA + kTileB)];     // A tiles [kS], then B tiles [kS]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % kWM, wn = wave / kWM;
  const long long M = N{km}, Nn = N{kn}, K = N{kk};
  // tiles, and workgroups, number less than 2^31 (the launcher's grid): 32-bit arithmetic, whose divisions are short
  const unsigned mt = (unsigned)((M + kBM - 1) / kBM), nt = (unsigned)((Nn + kBN - 1) / kBN);
  unsigned total = mt * nt;
  {' '.join(f'total *= (unsigned)N{self.atom(a)};' for a in g.batch)}
  // workgroups go to the 8 XCDs round-robin: each XCD takes a contiguous run of tiles (n fastest), so the
  // workgroups resident on it share rows of A and columns of B in its L2
  const unsigned parts = LFG_SPLIT ? (unsigned)p.n[{g.flags_at + 3}] : 1, per_xcd = (total * parts + 7) / 8;
  unsigned t = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (blockIdx.x >> 3 >= per_xcd || t >= total * parts) return;
  const unsigned part = LFG_SPLIT ? t / total : 0;      // slowest: neighbouring tiles of one part share rows of A or columns of B
  if (LFG_SPLIT) t -= part * total;
  // inside a batch element the tiles run in bands of kBand tile rows, column by column: the workgroups resident
  // on an XCD at a time (32 or 64 consecutive tiles) then cover a block of the output that is a few tiles tall and
  // wide, and read correspondingly few rows of A and columns of B past its L2
  constexpr unsigned kBand = kNT <= 256 ? 8 : 4;
  const unsigned element = {'t / (mt * nt)' if g.batch else '0'};      // of the batch
  t -= element * (mt * nt);
  const unsigned band = (unsigned)min(kBand * (unsigned long long)nt, 0xffffffffull), first = t / band * kBand, at = t % band;
  const unsigned tall = min(mt - first, kBand), tm = first + at % tall, tn = at / tall;
  {'long long blk = element;' if g.batch else ''}
  {' '.join(batch_decode)}
  const long long m0 = (long long)tm * kBM, n0 = (long long)tn * kBN;
  const {elem}* A = {a_base};
  const {elem}* B = {b_base};
  // this thread's pieces of a tile: byte offset at k = 0 and how many k are left from the piece's own k (0: the
  // piece lies outside the operand and is asked for beyond the buffer's range, i.e. arrives as zeros)
  const lfg_u32x4 rs_a = lfg_make_buffer(A, (unsigned)p.n[{g.flags_at + 1}]), rs_b = lfg_make_buffer(B, (unsigned)p.n[{g.flags_at + 2}]);
  unsigned offa[kPA], offb[kPB];
  int rooma[kPA], roomb[kPB];
#pragma unroll
  for (int j = 0; j < kPA; ++j) {{
    const int idx = tid + kNT * j;
    const long long oa = m0 + LfgPiece<a_rows, kBM>::outer(idx);
    const int ka = LfgPiece<a_rows, kBM>::k(idx);
    offa[j] = (unsigned)(2 * (oa * S{sam} + ka * S{sak}));
    rooma[j] = oa < M ? (int)min(K - ka, (long long)0x7fffffff) : 0;
  }}
#pragma unroll
  for (int j = 0; j < kPB; ++j) {{
    const int idx = tid + kNT * j;
    const long long ob = n0 + LfgPiece<b_rows, kBN>::outer(idx);
    const int kb = LfgPiece<b_rows, kBN>::k(idx);
    offb[j] = (unsigned)(2 * (ob * S{sbn} + kb * S{sbk}));
    roomb[j] = ob < Nn ? (int)min(K - kb, (long long)0x7fffffff) : 0;
  }}
  const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) const void*)lds;
  const unsigned stepa = (unsigned)(2 * {BK} * S{sak}), stepb = (unsigned)(2 * {BK} * S{sbk});
  const int steps = (int)((K + {BK - 1}) / {BK});
  const int st_begin = LFG_SPLIT ? (int)part * (int)p.n[{g.flags_at + 4}] : 0;
  const int st_end = LFG_SPLIT ? min(st_begin + (int)p.n[{g.flags_at + 4}], steps) : steps;
  // With few rows of A the loads of B from memory are the time.  There a workgroup's walk over k starts at a step of its
  // own, by tile column: with k contiguous and K a power of two every row of a step's window lies on the same few memory
  // channels, and workgroups that walk k in step all ask those (M 64, N 4096, K 16384: 39 -> 33 us; from M 512 on, where
  // matrix work is the time and tile columns share rows of A in an L2, it costs 4 ... 8 %).
  const int nsteps = st_end - st_begin;
  int ld_st = st_begin + (M <= 256 ? (int)(tn % (unsigned)nsteps) : 0), ld_left = nsteps;
  // A step's tiles, one wave-level load at a time (load j of kPA + kPB into buffer `buf`); past the last step the loads go
  // out against nothing, so that the number in flight behind a stage is always the same
  int k0 = ld_st * {BK};
  auto issue = [&](int buf, int j) {{
    if (j < kPA)
      lfg_dma<false>(rs_a, k0 < rooma[j] ? offa[j] + (unsigned)ld_st * stepa : 0xffffffffu,
                     lds0 + 2u * (unsigned)(kTileA * buf) + 1024u * (unsigned)(wave + kWaves * j));
    else
      lfg_dma<LFG_B_NT != 0>(rs_b, k0 < roomb[j - kPA] ? offb[j - kPA] + (unsigned)ld_st * stepb : 0xffffffffu,
                             lds0 + 2u * (unsigned)(kS * kTileA + kTileB * buf) + 1024u * (unsigned)(wave + kWaves * (j - kPA)));
  }};
  auto advance = [&]() {{
    if (++ld_st == st_end) ld_st = st_begin;
    k0 = --ld_left > 0 ? ld_st * {BK} : 0x7fffffff;
  }};
  lfg_f32x16 acc[kMB][kNB];
#pragma unroll
  for (int x = 0; x < kMB; ++x)
#pragma unroll
    for (int y = 0; y < kNB; ++y)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[x][y][i] = 0.0f;
  // operand f of step-of-16 ks of the stage in buffer `buf`: the kMB blocks of A (lane = m), then the kNB of B (lane = n:
  // the A operand of C^T = B^T A^T)
  constexpr int kF = kMB + kNB, kMF = kMB * kNB, kP = kPA + kPB, kKS = {BK // 16};
  auto operand = [&](int buf, int ks, int f) -> lfg_u32x4 {{
    if (f < kMB) return lfg_operand<a_rows, kBM>(&lds[kTileA * buf], kMB * wm + f, ks, lane);
    return lfg_operand<b_rows, kBN>(&lds[kS * kTileA + kTileB * buf], kNB * wn + f - kMB, ks, lane);
  }};
  // The operands of a step of 16 are read during the MFMAs of the one before, across stages too, so that no MFMA waits for a
  // read just issued.  The barrier of a stage stands in front of its last 16: by then every wave has read them, the next stage
  // has landed, and the loads of the stage kS on go out into this one's buffer between those MFMAs.  Against a barrier at the
  // end of a stage with its reads behind it, same tile, in a loop of its own: 8192^3 l 866 -> 829 us (1.33 PFLOP/s), m 1009 ->
  // 950; M 1024, N 4096, K 16384 m in 2 parts 133 -> 127.  What bounds it: matrix work at the clock it gets (large M); with few
  // rows of A the loads, which return in order per CU, so that A's, from L2, take their time beside B's from memory: 256 x
  // 16384 x 4096 d 39 us of loads alone (24 B's, 11 A's), 19 of products alone, 43 together.
#pragma unroll
  for (int s = 0; s < kS; ++s) {{
#pragma unroll
    for (int j = 0; j < kP; ++j) issue(s, j);
    advance();
  }}
  LFG_STAGE_BARRIER((kS - 1) * kP);
  lfg_u32x4 fr[2][kF];
#pragma unroll
  for (int f = 0; f < kF; ++f) fr[0][f] = operand(0, 0, f);
  int cur = 0;
  for (int i = 0; i < nsteps; ++i) {{
    const int next = cur == kS - 1 ? 0 : cur + 1;
#pragma unroll
    for (int ks = 0; ks < kKS; ++ks) {{
      if (ks == kKS - 1) LFG_STAGE_BARRIER((kS - 2) * kP);
#pragma unroll
      for (int j = 0; j < kMF; ++j) {{
#pragma unroll
        for (int f = j * kF / kMF; f < (j + 1) * kF / kMF; ++f)
          fr[(ks + 1) & 1][f] = ks < kKS - 1 ? operand(cur, ks + 1, f) : operand(next, 0, f);
        const int x = j / kNB, y = j % kNB;
        acc[x][y] = lfg_mfma(({elem})0.0f, fr[ks & 1][kMB + y], fr[ks & 1][x], acc[x][y]);
        if (ks == kKS - 1) {{
#pragma unroll
          for (int l = j * kP / kMF; l < (j + 1) * kP / kMF; ++l) issue(cur, l);
        }}
        __builtin_amdgcn_sched_barrier(0);
      }}
    }}
    advance();
    cur = next;
  }}
  // the loads against nothing still write zeros, and the last operands read are of such a stage: nothing may be left of
  // either when the LDS changes its role or is given back
  LFG_STAGE_BARRIER(0);
#if LFG_SPLIT
  // partials in accumulator order: [part][tile][wave][32 x 32 block][4][64 lanes] x 4 floats, every store 1 KB in a row
  float* ws = reinterpret_cast<float*>(p.ptr[{g.ws_ptr}]) +
              ((part * (long long)total + (long long)element * (mt * nt)) + (long long)tm * nt + tn) * (kBM * kBN) + wave * (kMB * kNB * 1024) + 4 * lane;
#pragma unroll
  for (int x = 0; x < kMB; ++x)
#pragma unroll
    for (int y = 0; y < kNB; ++y)
      if (m0 + 32 * (kMB * wm + x) < M && n0 + 32 * (kNB * wn + y) < Nn) {{
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *reinterpret_cast<lfg_f32x4*>(&ws[((x * kNB + y) * 4 + q) * 256]) =
              lfg_f32x4{{acc[x][y][4 * q], acc[x][y][4 * q + 1], acc[x][y][4 * q + 2], acc[x][y][4 * q + 3]}};
      }}
#else
  const bool row_stores = p.n[{g.flags_at}] != 0;
  // acc[x][y][i] = C[m][n], m = 32 * (kMB * wm + x) + lane % 32, n = 32 * (kNB * wn + y) + 8 * (i / 4) + 4 * (lane / 32) + i % 4.
  // Two n blocks at a time through the wave's own part of LDS ([32 * kMB m][64 n] fp32, 16-byte pieces permuted by the
  // row): afterwards a lane holds four consecutive n of one m and 16 neighbouring lanes cover 64 consecutive n.
  float* mine = reinterpret_cast<float*>(lds) + wave * (kMB * 2048);
  {lambdas}
  auto out_at = [&](long long i{km}, long long i{kn}) -> long long {{ return {ooff}; }};
#pragma unroll
  for (int pass = 0; pass < kNB / 2; ++pass) {{
    if (pass) __syncthreads();
    {{
      const int l32 = lane & 31, gg = lane >> 5;
#pragma unroll
      for (int x = 0; x < kMB; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
          for (int q = 0; q < 4; ++q) {{
            const int row = 32 * x + l32, piece = 8 * y + 2 * q + gg;
            const lfg_f32x16& c = acc[x][2 * pass + y];
            *reinterpret_cast<lfg_u32x4*>(&mine[row * 64 + 4 * (piece ^ (row & 15))]) =
                __builtin_bit_cast(lfg_u32x4, lfg_f32x4{{c[4 * q], c[4 * q + 1], c[4 * q + 2], c[4 * q + 3]}});
          }}
    }}
    __syncthreads();
#pragma unroll 4
    for (int j = 0; j < 8 * kMB; ++j) {{
      const int row = 4 * j + (lane >> 4), piece = lane & 15;
      const lfg_f32x4 c = __builtin_bit_cast(lfg_f32x4, *reinterpret_cast<const lfg_u32x4*>(&mine[row * 64 + 4 * (piece ^ (row & 15))]));
      const long long m = m0 + 32 * kMB * wm + row, n = n0 + 32 * kNB * wn + 64 * pass + 4 * piece;
      if (m < M && n < Nn) {{
        float r[4], rd[4][kRd];
#pragma unroll
        for (int e = 0; e < 4; ++e) read(rd[e], m, n + e < Nn ? n + e : n);
#pragma unroll
        for (int e = 0; e < 4; ++e) r[e] = epilogue(c[e], rd[e], m, n + e < Nn ? n + e : n);
        if (row_stores && n + 3 < Nn) {{
          lfg_st4<{out_t}>(p.ptr[{o}], out_at(m, n), r);
        }} else {{
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e < Nn) lfg_st<{out_t}>(p.ptr[{o}], out_at(m, n + e), r[e]);
        }}
      }}
    }}
  }}
#endif
}}
"""
        g.sum_source = f"""
// The parts of a 32 x 32 block of the output, one block per workgroup, added in fp32 in the order of k, and the epilogue on
// the sum.  Bound by its reads (written just before, mostly still in the last-level cache): a wave takes 8 rows x 32
// columns, so that it reads whole 128-byte lines and writes 64-byte pieces of rows.
extern "C" __global__ void __launch_bounds__(256) {self.name}_sum(const LfGenParams p) {{
  {' '.join(defs)}
  constexpr int kWM = LFG_WGM, kWN = LFG_WGN, kMB = LFG_MB, kNB = LFG_NB;
  constexpr int kBM = 32 * kWM * kMB, kBN = 32 * kWN * kNB;
  const long long M = N{km}, Nn = N{kn};
  const long long mt = (M + kBM - 1) / kBM, nt = (Nn + kBN - 1) / kBN;
  const unsigned mb = (unsigned)((M + 31) / 32), nb = (unsigned)((Nn + 31) / 32);   // at most the grid, which has 31 bits
  long long total = mt * nt;
  {' '.join(f'total *= N{self.atom(a)};' for a in g.batch)}
  const int bn = (int)(blockIdx.x % nb), bm = (int)(blockIdx.x / nb % mb);
  long long blk = blockIdx.x / nb / mb;
  const int tm = bm / (kWM * kMB), wm = bm / kMB % kWM, x = bm % kMB, tn = bn / (kWN * kNB), wn = bn / kNB % kWN, y = bn % kNB;
  const int lane = threadIdx.x & 63, row = 8 * (threadIdx.x >> 6) + (lane & 7), q = lane >> 4, gg = (lane >> 3) & 1;
  const float* ws = reinterpret_cast<const float*>(p.ptr[{g.ws_ptr}]) + ((blk * mt + tm) * nt + tn) * (kBM * kBN) +
                    (wm + kWM * wn) * (kMB * kNB * 1024) + ((x * kNB + y) * 4 + q) * 256 + 4 * (32 * gg + row);
  const long long m = 32 * bm + row, n = 32 * bn + 8 * q + 4 * gg, stride = total * (kBM * kBN);
  {' '.join(batch_decode)}
  if (m >= M || n >= Nn) return;
  {lambdas}
  float r[4], rd[4][kRd];
#pragma unroll
  for (int e = 0; e < 4; ++e) read(rd[e], m, n + e < Nn ? n + e : n);
  lfg_f32x4 c = {{0.0f, 0.0f, 0.0f, 0.0f}};
  const int parts = (int)p.n[{g.flags_at + 3}];
  for (int z = 0; z < parts; z += 4) {{
    lfg_f32x4 t[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) t[u] = *reinterpret_cast<const lfg_f32x4*>(&ws[min(z + u, parts - 1) * stride]);
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (z + u < parts) c += t[u];
  }}
  auto out_at = [&](long long i{km}, long long i{kn}) -> long long {{ return {ooff}; }};
#pragma unroll
  for (int e = 0; e < 4; ++e) r[e] = epilogue(c[e], rd[e], m, n + e < Nn ? n + e : n);
  if (p.n[{g.flags_at}] != 0 && n + 3 < Nn) {{
    lfg_st4<{out_t}>(p.ptr[{o}], out_at(m, n), r);
  }} else {{
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < Nn) lfg_st<{out_t}>(p.ptr[{o}], out_at(m, n + e), r[e]);
  }}
}}
"""
        return Kernel(self.name, src, self.bufs, self.atoms, self.strides, self.scalars, par)



# us per step of 64 k with every CU busy (s, n: up to 256 workgroups, one per CU, and beyond), us per workgroup besides (first
# loads, results), workgroups resident at a time
_COST = {"s": ((0.65, 1.01), 7.0, 512), "d": ((0.53, 0.53), 7.4, 256), "m": ((0.84, 0.84), 8.2, 256),
         "l": ((1.38, 1.38), 9.5, 256), "n": ((0.46, 0.94), 5.2, 512)}


@functools.lru_cache(maxsize=4096)
def choose(M: int, N: int, K: int, batch: int) -> tuple:
    """(tile shape, parts that k is split into) of a product: the candidate with the least time in a model of rounds of
    resident workgroups, plus, for a split product, the sum's launch and the traffic of its partials.  The model's constants
    are fitted to every candidate on 42 shapes (M 16 ... 8192, N 640 ... 16384, K 512 ... 16384, weights from HBM); there the
    choice is within 3 % of the best on 39, the others are 5 % (777 x 3000, K 5000), 10 % (6388 x 2880, K 1472, with gelu: m 98.9,
    s 90.3 us) and 7 % off (100 x 1024, K 4096: n in 13 parts 12.6, in 8 11.8).  What it is for: a product whose tiles leave
    most CUs idle, or alone with the latency of their loads.  M 256, us: N 4096 K 16384 218 (64 tiles s) -> 49 (d, 4 parts);
    N 16384 K 4096 66 -> 46 (d); M 64, N 4096 K 16384 214 -> 29 (n, 8 parts); M 1024, N 4096 K 16384 218 -> 130 (l, 4 parts);
    M 2000, N 1024 K 512 17 -> 11 (n).  n serves the fewest rows too: its tile pads least.  M up to 32, d or
    s / n, us: 16 x 4096, K 4096 13.5 / 12.7; 32 x 1024, K 4096 11.0 / 10.0; 8 x 4096, K 16384 29.4 / 26.3; 3 x 21888, K 3456 35.2 / 29.5; of
    99 drawn products, batches of 1 ... 16, 0.93 of the time in the mean, two are 4 % slower."""
    steps = -(-K // BK)
    best, best_t = ("s", 1), math.inf
    for shape, ((step_1, step_2), fixed, slots) in _COST.items():
        bm, bn = tile_extent(shape)
        if shape in "ml" and M <= bm // 2 or shape == "l" and N <= bn // 2:
            continue                         # half of the tile would be padding, and a smaller one has less (s, d, n)
        tiles = -(-M // bm) * -(-N // bn) * batch
        for parts in range(1, max(1, min(32, steps // 4)) + 1):
            if parts > 1 and tiles * parts > slots:      # one round, whose partials are 2^24 floats at most
                break
            per_part = -(-steps // parts)
            rounds, rest = divmod(tiles * parts, slots)
            t = rounds * (per_part * step_2 + fixed)
            if rest:
                t += per_part * (step_1 if rest <= 256 else step_2) + fixed
            if parts > 1:
                t += 1.1 + 0.087 * parts + parts * M * N * batch * 8 / 5.8e6
            if t < best_t:
                best, best_t = (shape, parts), t
    return best


def stream_b(M: int, N: int, K: int, own: int, shared: int) -> bool:
    """B by non-temporal loads (16-bit elements; ``own``, ``shared`` of ``b_batches``): they leave an L2 to A, and cost where several
    tiles read B at different times, or where it would have stayed in a cache.
    Non-temporal over plain, 160 drawn steps linear -> gelu -> linear, weights of other layers in between: 17 ... 128 rows 1.00 ... 1.10 (mean 1.04)
    below 50 MB, 0.98 from there to 100, 0.94 beyond; 129 ... 256 rows 1.06 below 50 MB, 1.03 up to 100, 0.97 beyond.  204 drawn single products:
    up to 16 rows 0.98 (0.95 from 50 MB on); 17 ... 64 rows 1.00 below 100 MB, 0.95 beyond; 65 ... 256 rows 1.04 below 100 MB, 1.01 beyond.  us,
    M x N x K, plain / non-temporal: 8 x 16384 x 4096 31.0 / 28.9, 64 x 28672 x 8192 83.5 / 74.2, 128 x 4096 x 4096 16.2 / 18.4, 256 x 4096 x 4096 22.4 /
    27.2, 256 x 2048 x 8192 22.3 / 26.1; linear -> gelu -> linear of 256 rows, 2048 / 8192 wide 45.2 / 48.6, 4096 / 16384 103.7 / 99.0.  A B that is
    still in a cache from the call before: 256 x 4096 x 4096 21.6 / 27.2, 256 x 16384 x 4096 46.5 / 48.3.
    Batches, B x M x N x K: shared weights 2 x 128 x 4096 x 4096 25.4 / 28.7, 4 x 16 x 16384 x 4096 76 / 87, 16 x 128 x 16384 x 4096 319 / 407;
    a B for each 64 x 64 x 512 x 512 11.4 / 10.7, 32 x 100 x 2048 x 2048 77 / 66, 16 x 256 x 1024 x 1024 19.1 / 19.2."""
    if shared > 1 or M > 256:
        return False
    return own > 1 or M <= 16 or 2 * N * K >= (48 << 20 if M <= 128 else 96 << 20)
