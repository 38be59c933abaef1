// lf_attn_bwd.hip — backward of the fused attention forward (dense K/V, mask none / causal /
// sliding window, scale, optional softcap; no bias) for gfx950.  The reference has no backward
// (its README lists it as future work); the formulas are the standard ones for
// O = softmax(scale * Q K^T + mask) V with the row log-sum-exp L kept by the forward:
//   P = exp(scale * Q K^T - L),  dV = P^T dO,  dP = dO V^T,  delta = rowsum(dO * O),
//   dS = scale * P * (dP - delta),  dQ = dS K,  dK = dS^T Q.
// With a softcap (LF_SOFTCAP) the scores are T = cap * tanh(scale * Q K^T / cap), P = exp(T - L), and
// dS picks up the derivative of the cap: dS = scale * (1 - tanh^2) * P * (dP - delta).
// Three kernels, no atomics, every result written once (deterministic):
//   lf_attn_bwd_delta : delta[b, h, q], in front of the other two unless lf_attn_bwd_dq has 256 threads and forms it itself
//                       (never with LF_BW_DS)
//   lf_attn_bwd_dq    : a workgroup owns 128 or 256 query rows of one (batch, head) -- 4 or 8 waves x
//                       32 rows, Q^T and dO^T in registers -- and walks the kv tiles (64 keys); with LF_BW_DS it
//                       reads the dS that lf_attn_bwd_dkdv has left instead of forming it, and runs behind it
//   lf_attn_bwd_dkdv  : a workgroup owns 64, 128 or 256 keys of one (batch, kv head) -- 4 waves x 32 or 64
//                       keys (64: two waves of keys, twice over), K^T and V^T of its keys in registers as MFMA B operands -- and walks the
//                       q tiles (64 rows) of the query heads of the group that can see them
// The tiles that are walked are kept in LDS once and read both ways: along their rows (ds_read_b128,
// rows of the tile = MFMA rows) and transposed (rows of the tile = MFMA k).  As in the forward, the accumulator of the first product is, as
// held, the B operand of the second, so P and dS never leave registers.
// L and the exponent are in log2 units (the forward writes L2 = offset + log2(sum)).

struct LfAttnBwdParams {
  const lf_elem* q;       // [B, Hq, Sq, D]
  const lf_elem* k;       // [B, Hkv, Sk, D]
  const lf_elem* v;
  const lf_elem* o;       // forward output
  const lf_elem* dout;    // gradient of the output
  lf_elem* dq;
  lf_elem* dk;
  lf_elem* dv;
  const float* lse;       // [B, Hq, Sq] row log-sum-exp of the scaled, masked scores, log2 units
  float* delta;           // [B, Hq, Sq] scratch: -rowsum(dO * O)
  long long q_sb, q_sh, q_ss;      // element strides (d stride 1)
  long long k_sb, k_sh, k_ss;
  long long v_sb, v_sh, v_ss;
  long long o_sb, o_sh, o_ss;
  long long do_sb, do_sh, do_ss;
  long long dq_sb, dq_sh, dq_ss;
  long long dk_sb, dk_sh, dk_ss;
  long long dv_sb, dv_sh, dv_ss;
  int B, Hq, Hkv, Sq, Sk;
  int window;
  float scale;
  float softcap;          // LF_SOFTCAP: cap of cap * tanh(s / cap)
  lf_elem* ds;            // LF_BW_DS: dS as lf_attn_bwd_dkdv leaves it for lf_attn_bwd_dq, lf_bw_ds_row below
  long long ds_sh;        // elements of it per (batch, query head)
};

#define LF_BW_NT 256
#ifndef LF_BW_GROUP
#define LF_BW_GROUP 4      /* (batch, kv head) pairs of one XCD whose workgroups are dispatched together */
#endif
// Is the score with (query - key) = t kept?  Callers fold the bound of the key sequence into t.
__device__ __forceinline__ bool lf_bw_keep(int t, int window) {
#if LF_MASK == 0
  (void)window;
  return t > -(1 << 29);
#elif LF_MASK == 1
  (void)window;
  return t >= 0;
#else
  return (unsigned)t < (unsigned)window;
#endif
}

#ifndef LF_BW_DS
#define LF_BW_DS 0         /* 1: lf_attn_bwd_dkdv leaves dS in memory, lf_attn_bwd_dq is the one product dQ = dS K */
#endif
// dS in memory: per (batch, query head) the 32 x 32 blocks (2 KB) that hold a visible score, those of 32 queries in a row in the
// order of their keys.  Blocks in front of block (qb, 0) of a head, nkb = key blocks; under a window a row starts at key
// block qb - (window + 30) / 32, which may lie before the first.
__device__ __forceinline__ int lf_bw_ds_row(int qb, int nkb, int window) {
#if LF_MASK == 0
  return qb * nkb;
#elif LF_MASK == 1
  const int m = min(qb, nkb);
  return m * (m + 1) / 2 + (qb - m) * nkb;
#else
  const int before = (window + 30) / 32;
  return qb * (before + 1) - (qb - before);
#endif
}
// A block holds what the lanes of lf_attn_bwd_dkdv hold as the B operand of dK^T += Q^T dS, 16-byte chunks (half h of the 32
// queries, lane half g, key) of 8 queries, permuted so that the transposed reads of lf_attn_bwd_dq (4 keys, all 16 queries
// of both halves at a time) touch every LDS bank once: byte offset of lane (g, key)'s chunk of half 0; half 1 is (it ^ 128) + 1024.
__device__ __forceinline__ unsigned lf_bw_ds_chunk(int key, int g) {
  return 16u * (unsigned)(32 * g + 16 * (key >> 4) + 4 * (((key >> 2) & 3) ^ g) + (key & 3));
}

// delta[row] = sum_d dO[row][d] * O[row][d]; 16 lanes per row, 8 elements per lane
extern "C" __global__ void __launch_bounds__(LF_BW_NT) lf_attn_bwd_delta(const LfAttnBwdParams p) {
  const long long row = (long long)blockIdx.x * (LF_BW_NT / 16) + threadIdx.x / 16;
  const int piece = threadIdx.x % 16;
  const long long nrows = (long long)p.B * p.Hq * p.Sq;
  float s = 0.0f;
  if (row < nrows && piece < LF_CPR) {
    const int qi = (int)(row % p.Sq);
    const int h = (int)((row / p.Sq) % p.Hq);
    const int b = (int)(row / ((long long)p.Sq * p.Hq));
    const lf_elem8 ov = *reinterpret_cast<const lf_elem8*>(p.o + b * p.o_sb + h * p.o_sh + qi * p.o_ss + 8 * piece);
    const lf_elem8 gv = *reinterpret_cast<const lf_elem8*>(p.dout + b * p.do_sb + h * p.do_sh + qi * p.do_ss + 8 * piece);
#pragma unroll
    for (int e = 0; e < 8; ++e) s += (float)ov[e] * (float)gv[e];
  }
  s += __shfl_xor(s, 1, 64);
  s += __shfl_xor(s, 2, 64);
  s += __shfl_xor(s, 4, 64);
  s += __shfl_xor(s, 8, 64);
  if (row < nrows && piece == 0) p.delta[row] = -s;
}

// wait for this wave's direct loads and LDS writes, then meet the other waves.  The wait is the
// builtin, not inline asm, so that the compiler's wait-counter pass sees that nothing is
// outstanding afterwards: otherwise it waits again inside the step -- for the operands loaded
// before the loop and before overwriting a register a tracked load wrote -- with vmcnt values
// that also drain the direct loads of the next stage just issued (0x0070: vmcnt(0) lgkmcnt(0))
#define LF_BW_BARRIER()                      \
  do {                                       \
    asm volatile("" ::: "memory");           \
    __builtin_amdgcn_s_waitcnt(0x0070);      \
    __builtin_amdgcn_s_barrier();            \
    asm volatile("" ::: "memory");           \
  } while (0)

// MFMAs of both product kernels with the register file of every operand spelled out.  At one wave per
// SIMD a kernel has 512 registers per lane, and the compiler then gives every MFMA an AGPR
// destination while keeping what it computes with in VGPRs: left to it, the loop carries hundreds
// of v_accvgpr moves per step.  Here dK^T / dV^T (written in the loop, read after it) and the
// loop-invariant K^T / V^T operands live in AGPRs, S^T / dP^T (read by the VALU right away) in VGPRs.
// What the compiler would otherwise see to: an MFMA result may be read 12 wait states after the MFMA
// was issued at the earliest (LF_BW_MFMA_DRAIN), and a VGPR written by the VALU may be an MFMA
// operand 2 wait states later (LF_BW_VALU_SETTLE); back-to-back MFMAs on one accumulator need nothing.
// What it cannot see to at all: a register copy or a spill of its own placed right behind one of these
// MFMAs would read the accumulator too early.  The live ranges are laid out so that it has no reason
// for either, and tests/test_kernel_codegen.py checks the generated code for it.
#if LF_DTYPE == 0
#define LF_BW_MFMA "v_mfma_f32_32x32x16_bf16"
#else
#define LF_BW_MFMA "v_mfma_f32_32x32x16_f16"
#endif
#define LF_BW_MFMA_DRAIN "s_nop 9\n\ts_nop 9"
#define LF_BW_MFMA_DRAIN_LAST "s_nop 15\n\ts_nop 15\n\ts_nop 15"     /* behind the last MFMAs issued: one may still wait for the pipe */
#define LF_BW_VALU_SETTLE "s_nop 1"
// c (VGPRs) = a (VGPRs) x b (AGPRs)
__device__ __forceinline__ void lf_bw_mfma_first(lf_f32x16& c, const lf_u32x4& a, const lf_u32x4& b) {
  asm volatile(LF_BW_MFMA " %0, %1, %2, 0" : "=&v"(c) : "v"(a), "a"(b));
}
// c (VGPRs) += a (VGPRs) x b (AGPRs)
__device__ __forceinline__ void lf_bw_mfma_vva(lf_f32x16& c, const lf_u32x4& a, const lf_u32x4& b) {
  asm volatile(LF_BW_MFMA " %0, %1, %2, %0" : "+v"(c) : "v"(a), "a"(b));
}
// accumulators X^T[d][n] (lane n = lane % 32; element i of block db is d = 32*db + 8*(i/4) + 4*g + i%4)
// -> rows 0 .. 31 of a [.., D] matrix, those below `valid`.  They meet in the wave's part of the LDS (`rows_lds`, LF_BW_ROWS_LDS
// bytes that nobody reads any more) and leave whole, neighbouring lanes with the pieces of one row, by non-temporal stores:
// 32-byte pieces of every lane's own row take the L2 from what the launch reads.
#ifndef LF_STAY
#define LF_STAY 0        /* 1: 32-byte pieces by plain stores all the same, which save the way through LDS and leave the gradients
                            nearer to whoever reads them next.  All backward launches, times whole over pieces, 57 shapes, alone / with an
                            element-wise kernel behind them that reads the gradients: dQ of 0.2 ... 10 MB 0.98 ... 1.04 / 0.99 ... 1.13 (0.4
                            MB, unmasked B5 H4 S163 D64 16.6 -> 16.8 and 27.1 -> 30.5 us), 10 ... 30 MB 0.95 ... 1.00 / 0.99 ... 1.03, above
                            0.90 ... 1.00 / 0.95 ... 1.01 (67 MB, causal B4 H32 S2048 D128 556 -> 535 and 618 -> 613, unmasked 885 -> 855
                            and 953 -> 906) (lowering.bwd_grads_stay) */
#endif
#define LF_BW_OUT_STRIDE (LF_D * 2 + 16)
#define LF_BW_ROWS_LDS (32 * LF_BW_OUT_STRIDE)
__device__ __forceinline__ void lf_bw_store_rows(const lf_f32x16* acc, unsigned rows_lds, lf_elem* rows, long long stride, int valid, int lane) {
  typedef __attribute__((address_space(3))) lf_u32x2* lds_write_t;
  typedef __attribute__((address_space(3))) const lf_u32x4* lds_read_t;
  const int l32 = lane & 31, g = lane >> 5;
#if LF_STAY
  (void)rows_lds;
  lf_elem* row = rows + l32 * stride + 8 * g;
#pragma unroll
  for (int db = 0; db < LF_NDB; ++db) {
    unsigned ch[4][2];
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      lf_elem4 w;
#pragma unroll
      for (int e = 0; e < 4; ++e) w[e] = lf_from_float(acc[db][4 * i4 + e]);
      const lf_u32x2 wu = __builtin_bit_cast(lf_u32x2, w);
      ch[i4][0] = wu[0];
      ch[i4][1] = wu[1];
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {      // halves of a row change lanes: 8 consecutive d's each, 32 contiguous bytes per row and store
      auto r0 = __builtin_amdgcn_permlane32_swap(ch[2 * j][0], ch[2 * j + 1][0], false, false);
      auto r1 = __builtin_amdgcn_permlane32_swap(ch[2 * j][1], ch[2 * j + 1][1], false, false);
      const lf_u32x4 out = {r0[0], r1[0], r0[1], r1[1]};
      if (l32 < valid) *reinterpret_cast<lf_u32x4*>(row + 32 * db + 16 * j) = out;
    }
  }
#else
  lf_wave_exchange();              // the rows before these have been read
#pragma unroll
  for (int db = 0; db < LF_NDB; ++db)
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      lf_elem4 w;
#pragma unroll
      for (int e = 0; e < 4; ++e) w[e] = lf_from_float(acc[db][4 * i4 + e]);
      *(lds_write_t)(size_t)(rows_lds + (unsigned)(l32 * LF_BW_OUT_STRIDE + 64 * db + 16 * i4 + 8 * g)) = __builtin_bit_cast(lf_u32x2, w);
    }
  lf_wave_exchange();
  constexpr int kRows = 64 / LF_CPR;
#pragma unroll
  for (int i = 0; i < 32 / kRows; ++i) {
    const int r = kRows * i + lane / LF_CPR, c = lane % LF_CPR;
    const lf_u32x4 x = *(lds_read_t)(size_t)(rows_lds + (unsigned)(r * LF_BW_OUT_STRIDE + 16 * c));
    if (r < valid) __builtin_nontemporal_store(x, reinterpret_cast<lf_u32x4*>(rows + r * stride + 8 * c));
  }
#endif
}

// ---- tiles that are kept in LDS once and read both ways.  A 64-row tile is row-major and unpadded; the 16-byte
// chunks of a row are permuted by an XOR with lf_bw_swz(row), the low bits of the row (counted in 256-byte bank
// spans) rotated so that both read patterns touch every bank once: 16 consecutive rows, one logical chunk
// (ds_read_b128, rows = MFMA rows) get 16 different values, and the 4 rows x 64 bytes of a transposed read differ in
// the bits above the two that its four chunks vary.  Against a copy per read pattern that is half the LDS and half
// the L2 -> LDS traffic, and leaves room for a third stage.
__device__ __forceinline__ int lf_bw_swz(int row) {
  const int r = row / LF_RPS;
#if LF_HEAD_DIM == 128
  return ((r & 3) << 2) | ((r >> 2) & 3);
#else
  return ((r & 1) << 2) | ((r >> 1) & 3);
#endif
}
#define LF_BW_ROWB (LF_D * 2)                       /* bytes per row of a tile */
#define LF_BW_TILEB (64 * LF_BW_ROWB)               /* bytes per tile */
typedef __attribute__((address_space(3))) const lf_u32x4* lf_bw_lds_u32x4;
typedef __attribute__((address_space(3))) lf_s16x4* lf_bw_lds_s16x4;
// This lane's offset for fragment (row block 0, 16-dim step 0) / (16-row step 0, 32-dim block 0); the other
// fragments are an XOR of address bits below the row size and a constant away (tile addresses are multiples of it).
__device__ __forceinline__ unsigned lf_bw_rm_off(int l32, int g) {
  return (unsigned)(l32 * LF_BW_ROWB + 16 * (g ^ lf_bw_swz(l32)));
}
__device__ __forceinline__ unsigned lf_bw_tr_off(int lane) {
  const int j = lane & 15, dh = (lane >> 4) & 1, row = 4 * (lane >> 5) + (j >> 2);
  return (unsigned)(row * LF_BW_ROWB + 16 * ((2 * dh + ((j & 3) >> 1)) ^ lf_bw_swz(row)) + 8 * (j & 1));
}
// base ^ bits.  Volatile, so that equal addresses of different reads are formed again instead of being kept: a stage has
// 24 of them and there are no registers to hold them in.
__device__ __forceinline__ unsigned lf_bw_flip(unsigned base, int bits) {
  if (bits == 0) return base;
  unsigned a;
  asm volatile("v_xor_b32 %0, %1, %2" : "=v"(a) : "i"(bits), "v"(base));
  return a;
}
// rows 32*blk + lane % 32, d = 16*ks + 8*g .. +7 of the tile `disp` bytes into a stage; `base` = LDS address of the
// stage + lf_bw_rm_off
__device__ __forceinline__ lf_u32x4 lf_bw_read_rm(unsigned base, int disp, int blk, int ks) {
  return *(lf_bw_lds_u32x4)(size_t)(lf_bw_flip(base, 32 * ks) + (unsigned)(disp + 32 * blk * LF_BW_ROWB));
}
// transposed: d = 32*db + lane % 32, rows 16*kk + 8*(s/4) + 4*g + s%4 for s = 0 .. 7; `base` = stage + lf_bw_tr_off
__device__ __forceinline__ lf_u32x4 lf_bw_read_tr(unsigned base, int disp, int kk, int db) {
  lf_u32x4 a;
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    const unsigned src = lf_bw_flip(base, 64 * db + 32 * half) + (unsigned)(disp + (16 * kk + 8 * half) * LF_BW_ROWB);
    const lf_u32x2 t = __builtin_bit_cast(lf_u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lf_bw_lds_s16x4)(size_t)src));
    a[2 * half] = t[0];
    a[2 * half + 1] = t[1];
  }
  return a;
}
// One direct load of a tile (NT threads: kRows whole rows per load of the workgroup): row row0 + srow + kRows * ps of
// the matrix behind `rs`; rows past its end arrive as zeros.  `lane_off` = lf_bw_load_off.
__device__ __forceinline__ unsigned lf_bw_load_off(unsigned rowb, int tid) {
  const int srow = tid / LF_CPR, sch = tid % LF_CPR;       // a load is a multiple of 16 rows: the swizzle repeats
  return (unsigned)srow * rowb + 16u * (unsigned)(sch ^ lf_bw_swz(srow));
}
template <int NT>
__device__ __forceinline__ void lf_bw_load_rows(const lf_u32x4& rs, unsigned rowb, int row0, unsigned tile, unsigned lane_off,
                                                int ps, int wave) {
  constexpr int kRows = NT / LF_CPR, kRowsPerWave = 64 / LF_CPR;
  static_assert(kRows % 16 == 0, "a load must keep the swizzle phase");
  lf_dma_to_lds_at(rs, (unsigned)(row0 + kRows * ps) * rowb + lane_off,
                   tile + (unsigned)((kRows * ps + kRowsPerWave * wave) * LF_BW_ROWB));
}

// One wave-level direct-to-LDS load of 64 floats: lane i's lands at lds_addr + 4 * i.
__device__ __forceinline__ void lf_dma_dword_to_lds_at(const lf_u32x4& rs, unsigned voff, unsigned lds_addr) {
  unsigned m0_written;
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tbuffer_load_dword %2, %3, 0 offen lds"
               : "={m0}"(m0_written) : "s"(lds_addr), "v"(voff), "s"(rs) : "memory");
}

// lf_dma_to_lds_at for bytes that are read once: they do not push what is shared out of the L2
__device__ __forceinline__ void lf_dma_nt_to_lds_at(const lf_u32x4& rs, unsigned voff, unsigned lds_addr) {
  unsigned m0_written;
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %3, 0 offen nt lds"
               : "={m0}"(m0_written) : "s"(lds_addr), "v"(voff), "s"(rs) : "memory");
}

// MFMAs with every operand in VGPRs (the accumulator: VGPRs); first of a chain: started from `c0`, or from zero.  The
// matrix core reads `c0` late: keep it alive (LF_BW_HOLD) until another MFMA has been issued behind its readers.
#define LF_BW_HOLD(c0) asm volatile("" :: "v"(c0))
__device__ __forceinline__ void lf_bw_mfma_vvv(lf_f32x16& c, const lf_u32x4& a, const lf_u32x4& b) {
  asm volatile(LF_BW_MFMA " %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
}
__device__ __forceinline__ void lf_bw_mfma_from(lf_f32x16& c, const lf_u32x4& a, const lf_u32x4& b, const lf_f32x16& c0) {
  asm volatile(LF_BW_MFMA " %0, %1, %2, %3" : "=&v"(c) : "v"(a), "v"(b), "v"(c0));
}
__device__ __forceinline__ void lf_bw_mfma_zero(lf_f32x16& c, const lf_u32x4& a, const lf_u32x4& b) {
  asm volatile(LF_BW_MFMA " %0, %1, %2, 0" : "=&v"(c) : "v"(a), "v"(b));
}

// c (AGPRs) += a x b (VGPRs), with the accumulator handed over as an input: the kernels keep up to all of their AGPRs in
// use from its first to its last instruction, and accumulators that the compiler sees change in the loop leave its
// register allocator without a free tuple to resolve a control-flow merge with -- it spills a thousand registers.  So
// it sees 16 values that are defined once, used throughout and defined anew by the drain behind the loop; they stay in
// their registers for lack of any other (tests/test_kernel_codegen.py holds the generated code to that).
__device__ __forceinline__ void lf_bw_mfma_hidden(const lf_f32x16& c, const lf_u32x4& a, const lf_u32x4& b) {
  asm volatile(LF_BW_MFMA " %0, %1, %2, %0" ::"a"(c), "v"(a), "v"(b));
}

#ifndef LF_BW_W
#define LF_BW_W 1        /* 32-key blocks per wave of lf_attn_bwd_dkdv: every fragment read from LDS feeds so many MFMAs */
#endif
#ifndef LF_BW_QSPLIT
#define LF_BW_QSPLIT 0   /* 1: two waves of keys instead of four, twice over: one pair takes the first 32 queries of a tile, one the others */
#endif
// s_waitcnt vmcnt: all but the newest kMost (and kMore beyond them, if there are that many)
template <int kMost, int kMore> __device__ __forceinline__ void lf_bw_wait(int more) {
  constexpr int kBoth = kMost + kMore;
  if (kMore > 0 && more == kMore) __builtin_amdgcn_s_waitcnt((kBoth & 15) | 0x70 | ((kBoth >> 4) << 14));
  else __builtin_amdgcn_s_waitcnt((kMost & 15) | 0x70 | ((kMost >> 4) << 14));
}
#ifndef LF_BW_PF
#define LF_BW_PF (LF_BW_W == 2 && LF_HEAD_DIM == 128 ? 3 : 4)   /* fragments read ahead of the MFMAs that take them (there, a fourth spills) */
#endif

#ifndef LF_BW_VL
#define LF_BW_VL (LF_BW_W == 2 && LF_HEAD_DIM == 128 ? 5 : 0)    /* 16-dim steps of the V^T operand kept in LDS instead of registers */
#endif

// dK and dV of 128 * LF_BW_W keys of one (batch, kv head): 4 waves, one per SIMD, wave w the keys 32 * LF_BW_W * w ...
// What bounds it: the four products' MFMAs and the power they draw.  At LF_BW_W = 2, D = 128 the 512 registers are spoken
// for (dK^T, dV^T 256 AGPRs, K^T / V^T operands 96 VGPRs with half of V^T in LDS, S^T and dP^T 64, P and dS 32, fragments 12)
// and an MFMA pair costs one LDS fragment read.  Causal bf16 B4 H32 S2048 D128: 390 us in the form before (a copy of each
// tile per read pattern, one MFMA per fragment, a wait in front of every group of probabilities), 298 us now = 0.98
// PFLOP/s executed at 0.39 of the MFMA cycles; without its LDS reads, direct loads, barrier and exponentials the same
// stream still takes three quarters of that, and the read-ahead (2 ... 8 fragments) makes no difference.
// Work of a wave: a stream of blocks of 32 queries, two per 64-query tile, and per block four phases of MFMAs whose
// A fragments come through one read-ahead ring that runs on into the next block:
//   S^T = Q K^T
//   dP^T = dO V^T                    accumulators start at -delta; P between these MFMAs
//   dV^T += dO^T P                   dS = P (dP - delta) between these
//   dK^T += Q^T dS
// L is subtracted in the exponent (one fused multiply-add, P = 2^(c S - L)), not by starting S at -L / c: there every step of
// the product rounds at the size of L / c (dV in fp16 at exponents of 1e5: 1.2e-3 off instead of 2.9e-4), a scale of 0 gives
// NaN, and it is no faster (all launches, us, started / subtracted: causal B4 H32 S2048 D128 538 / 537, B8 16/4 S1000 D64
// 129 / 127, unmasked B2 32/8 S4096 1627 / 1618, softcap B4 32/8 S2048 631 / 628).
// Three LDS stages: a tile's loads are issued in the second half of the step two before its own, and the one barrier per
// step, in its middle, says both that the next tile has landed and that the tile before this one is free.
// With LF_BW_QSPLIT a workgroup owns 64 keys, 32 per wave, every key held by two waves: one pair walks the first 32 queries of each
// tile, the other the last, and their sums meet in LDS at the end.  A tile is then one block per wave: its barrier stands in
// front of the block and waits for loads issued two blocks before, which takes a fourth stage.  For launches of few
// workgroups (lowering.bwd_q_split): causal D64 B8 16/4 S1000, 256 workgroups of 128 keys whose longest walks twice the mean,
// 89 -> 60 us.
// With LF_BW_DS the B operands dS also leave for memory, two stores per 32 x 32 block between the MFMAs that take them, and the
// barrier does not wait for them: 297 -> 340 us of the above for 545 MB (352 with plain stores, which take L2 from Q and dO).
extern "C" __global__ void __launch_bounds__(LF_BW_NT, 1) lf_attn_bwd_dkdv(const LfAttnBwdParams p) {
  constexpr int KB = LF_BW_W, kKeyWaves = LF_BW_QSPLIT ? 2 : 4, kStages = LF_BW_QSPLIT ? 4 : 3;
  constexpr int kKeys = 32 * KB * kKeyWaves;
  __shared__ __attribute__((aligned(256))) lf_elem tiles[kStages][2][64 * LF_D];        // Q, dO
  __shared__ __attribute__((aligned(16))) float stats[kStages][2][64];                  // of the 64 rows: L, start of dP
#if LF_BW_VL
  __shared__ lf_u32x4 v_lds[LF_BW_VL][KB][LF_BW_NT];                               // V^T operands that the registers have no room for
#endif

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31;
  const int g = lane >> 5;

  const int nkt = (p.Sk + kKeys - 1) / kKeys;
  // All key blocks of a (batch, kv head) share the Q / dO tiles they walk in one XCD's L2; the first key
  // block has the most steps under a causal mask.
  int bhkv, kt;
  if (!lf_slot_of_block(blockIdx.x, p.B * p.Hkv, nkt, LF_BW_GROUP, bhkv, kt)) return;
  const int hkv = bhkv % p.Hkv;
  const int b = bhkv / p.Hkv;
  const int group = p.Hq / p.Hkv;
  const int key0 = kKeys * kt + 32 * KB * (wave % kKeyWaves);    // first key of this wave
  const int my_qb = wave / kKeyWaves;                            // LF_BW_QSPLIT: the wave's 32 queries of a tile
  const int klast = min(key0 + 32 * KB, p.Sk) - 1;
  const int nqt = (p.Sq + 63) / 64;

  // K^T and V^T of this lane's keys as B operands (d = 16*ks + 8*g .. +7)
  constexpr int kVReg = LF_NKS - LF_BW_VL;
  lf_u32x4 kf[KB][LF_NKS], vf[KB][kVReg];
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
    const int kr = min(key0 + 32 * kb + l32, p.Sk - 1);
    const lf_elem* krow = p.k + (long long)b * p.k_sb + (long long)hkv * p.k_sh + (long long)kr * p.k_ss;
    const lf_elem* vrow = p.v + (long long)b * p.v_sb + (long long)hkv * p.v_sh + (long long)kr * p.v_ss;
#pragma unroll
    for (int ks = 0; ks < LF_NKS; ++ks) {
      kf[kb][ks] = *reinterpret_cast<const lf_u32x4*>(krow + 16 * ks + 8 * g);
      const lf_u32x4 x = *reinterpret_cast<const lf_u32x4*>(vrow + 16 * ks + 8 * g);
      if (ks < kVReg) vf[kb][ks] = x;
#if LF_BW_VL
      else v_lds[ks - kVReg][kb][tid] = x;
#endif
    }
  }
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
#pragma unroll
    for (int ks = 0; ks < LF_NKS; ++ks) asm volatile("" : "+v"(kf[kb][ks]));
#pragma unroll
    for (int ks = 0; ks < kVReg; ++ks) asm volatile("" : "+v"(vf[kb][ks]));
  }
#if LF_SOFTCAP
  const float sc_exp = p.scale / p.softcap * (2.0f * LF_LOG2E);   // 2^(s * sc_exp) = e^(2x)
  const float cexp = p.softcap * LF_LOG2E;                        // exponent of P: tanh x * cexp - L
#else
  const float cexp = p.scale * LF_LOG2E;                          // exponent of P: s * cexp - L
#endif

  lf_f32x16 dk[KB][LF_NDB], dv[KB][LF_NDB];
#pragma unroll
  for (int kb = 0; kb < KB; ++kb)
#pragma unroll
    for (int db = 0; db < LF_NDB; ++db) {
#pragma unroll
      for (int i = 0; i < 16; ++i) dk[kb][db][i] = dv[kb][db][i] = 0.0f;
      asm volatile("" : "+a"(dk[kb][db]), "+a"(dv[kb][db]));
    }

  // q tiles (64 rows) that hold a query seeing one of the workgroup's keys
  int qt_begin = 0, qt_end = nqt;
#if LF_MASK >= 1
  qt_begin = kKeys * kt / 64;                                   // q >= key
#endif
#if LF_MASK == 2
  qt_end = min(nqt, (min(kKeys * kt + kKeys, p.Sk) - 1 + p.window - 1) / 64 + 1);   // q - key < window
#endif
  // the steps of this workgroup: query heads of the group x q tiles, one flat sequence
  const int ntq = max(qt_end - qt_begin, 0);
  const int nsteps = group * ntq;

  const unsigned q_bytes = (unsigned)(((long long)(p.Sq - 1) * p.q_ss + LF_D) * 2);
  const unsigned g_bytes = (unsigned)(((long long)(p.Sq - 1) * p.do_ss + LF_D) * 2);
  const unsigned q_rowb = (unsigned)p.q_ss * 2u, g_rowb = (unsigned)p.do_ss * 2u;
  const unsigned q_loff = lf_bw_load_off(q_rowb, tid), g_loff = lf_bw_load_off(g_rowb, tid);
  constexpr int kPasses = 64 * LF_CPR / LF_BW_NT;      // loads of a wave per tile
  constexpr int kLoads = 2 * kPasses;
  const unsigned lds0 = lf_lds_addr(tiles);
  auto q_tile = [&](int st) { return lds0 + (unsigned)(2 * st * LF_BW_TILEB); };
  auto g_tile = [&](int st) { return lds0 + (unsigned)((2 * st + 1) * LF_BW_TILEB); };

  // ---- what is loaded next: query head, q tile; past the last step the loads go out against an empty range.  Waves 0
  // and 1 also bring the row statistics, L and -delta; those of rows past Sq are zeros: P is 1 there
  // and meets dO = 0.
  int ld_step = 0, ld_tile = qt_begin, ld_q0 = 0;
  const lf_elem* ld_q = p.q + (long long)b * p.q_sb + (long long)(hkv * group) * p.q_sh;
  const lf_elem* ld_g = p.dout + (long long)b * p.do_sb + (long long)(hkv * group) * p.do_sh;
  const float* ld_stat = (wave == 0 ? p.lse : p.delta) + ((long long)b * p.Hq + hkv * group) * p.Sq;
  lf_u32x4 q_rs, g_rs, stat_rs;
  auto aim = [&]() {
    const bool real = ld_step < nsteps;
    ld_q0 = 64 * ld_tile;
    q_rs = lf_make_buffer(ld_q, real ? q_bytes : 0u);
    g_rs = lf_make_buffer(ld_g, real ? g_bytes : 0u);
    stat_rs = lf_make_buffer(ld_stat, real && wave < 2 ? (unsigned)p.Sq * 4u : 0u);
    ++ld_step;
    if (++ld_tile == qt_end) {
      ld_tile = qt_begin;
      ld_q += p.q_sh;
      ld_g += p.do_sh;
      ld_stat += p.Sq;
    }
  };
  const unsigned stat0 = lf_lds_addr(stats);
  auto issue = [&](int st, int j) {      // load j of kLoads
    if (j < kPasses) lf_bw_load_rows<LF_BW_NT>(q_rs, q_rowb, ld_q0, q_tile(st), q_loff, j, wave);
    else lf_bw_load_rows<LF_BW_NT>(g_rs, g_rowb, ld_q0, g_tile(st), g_loff, j - kPasses, wave);
    if (j == kLoads - 1 && wave < 2)
      lf_dma_dword_to_lds_at(stat_rs, (unsigned)(ld_q0 + lane) * 4u, stat0 + (unsigned)((2 * st + wave) * 256));
  };
  // statistic `which` of the queries of block qb in accumulator order: element 4*i4 + e is query 32*qb + 8*i4 + 4*g + e
  const int stat_at = 4 * g + 32 * my_qb;
  auto read_stat4 = [&](int st, int which, int qb, int i4) {
    return *reinterpret_cast<const lf_f32x4*>(&stats[st][which][32 * qb + 8 * i4 + stat_at]);
  };
  auto read_stats = [&](int st, int which, int qb) {
    lf_f32x16 r;
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      const lf_f32x4 x = read_stat4(st, which, qb, i4);
#pragma unroll
      for (int e = 0; e < 4; ++e) r[4 * i4 + e] = x[e];
    }
    return r;
  };

  unsigned rm_off = lf_bw_rm_off(l32, g) + (unsigned)(32 * my_qb * LF_BW_ROWB), tr_off = lf_bw_tr_off(lane) + (unsigned)(32 * my_qb * LF_BW_ROWB);
  asm volatile("" : "+v"(rm_off), "+v"(tr_off));
  constexpr int NS = LF_NKS, NT = 2 * LF_NDB, NF = 2 * NS + 2 * NT;     // fragments of a block
  static_assert(kLoads <= NS, "a block's loads go out during its first two phases");
  static_assert(LF_BW_PF <= NS, "the read-ahead of a block's first phase");
  // fragment i of block qb of the stage: Q rows, dO rows, dO^T, Q^T
  auto frag = [&](int st, int qb, int i) {
    const unsigned sb = q_tile(st);
    if (i < NS) return lf_bw_read_rm(sb + rm_off, 0, qb, i);
    if (i < 2 * NS) return lf_bw_read_rm(sb + rm_off, LF_BW_TILEB, qb, (i - NS + kVReg) % NS);      // steps of V^T in LDS first
    const int j = i - 2 * NS;
    if (j < NT) return lf_bw_read_tr(sb + tr_off, LF_BW_TILEB, 2 * qb + j / LF_NDB, j % LF_NDB);
    return lf_bw_read_tr(sb + tr_off, 0, 2 * qb + (j - NT) / LF_NDB, j % LF_NDB);
  };
  lf_u32x4 pre[LF_BW_PF];            // the next block's first fragments
  auto read_ahead = [&](int st, int qb) {
#pragma unroll
    for (int f = 0; f < LF_BW_PF; ++f) pre[f] = frag(st, qb, f);
  };

  int ds_young = 0;                // LF_BW_DS: stores of this wave behind its last direct loads
#if LF_BW_DS
  const int nkb = (p.Sk + 31) / 32;
  lf_elem* ds_head = p.ds + ((long long)b * p.Hq + hkv * group) * p.ds_sh;      // of the query head that is walked
  unsigned ds_off = lf_bw_ds_chunk(l32, g);
  asm volatile("" : "+v"(ds_off));
#endif

  // One block of a wave: 32 queries (qb of stage st, first one q0) x its keys.  `loads`: those of stage `ld` are
  // issued between the MFMAs; the block read ahead is (st_n, qb_n).
  auto block = [&](const int qb, int st, int q0, const bool masked, const bool loads, int ld, int st_n, const int qb_n) {
    lf_u32x4 fr[NF + LF_BW_PF];
#pragma unroll
    for (int f = 0; f < LF_BW_PF; ++f) fr[f] = pre[f];
    lf_f32x16 s[KB], dp[KB], dinit;
    lf_f32x4 lse4[4];                // L of elements 4*i4 .. +3, read one group ahead of its first use
    lf_u32x4 pf[KB][2], dsf[KB][2];
#if LF_BW_VL
    lf_u32x4 vl[LF_BW_VL][KB];
#endif
    int rel[KB];                     // query minus key of element 0; a key past Sk fails every test
    if (masked) {
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        const int my_key = key0 + 32 * kb + l32;
        rel[kb] = my_key < p.Sk ? q0 + 4 * g - my_key : -(1 << 30);
        asm volatile("" : "+v"(rel[kb]));      // formed per block: what derives from it is not kept over the loop
      }
    }
    // P of elements 4*i4 .. +3 of key block kb; kept in fp32 in s for dS (with a cap: times its derivative)
    auto soft4 = [&](int kb, int i4) {
      lf_elem4 pw;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = 4 * i4 + e;
#if LF_SOFTCAP
        const float r = __builtin_amdgcn_rcpf(1.0f + lf_exp2(s[kb][i] * sc_exp));     // 1 / (e^(2x) + 1), x = s * scale / cap
        float pv = lf_exp2((1.0f - 2.0f * r) * cexp - lse4[i4][e]);
        const float dcap = 4.0f * r * (1.0f - r);                                      // 1 - tanh^2
#else
        float pv = lf_exp2(s[kb][i] * cexp - lse4[i4][e]);
#endif
        if (masked) {
          pv = lf_bw_keep(rel[kb] + 8 * i4 + e, p.window) ? pv : 0.0f;
        }
        pw[e] = lf_from_float(pv);
#if LF_SOFTCAP
        s[kb][i] = pv * dcap;
#else
        s[kb][i] = pv;
#endif
      }
      const lf_u32x2 pu = __builtin_bit_cast(lf_u32x2, pw);
      pf[kb][i4 / 2][2 * (i4 % 2)] = pu[0];
      pf[kb][i4 / 2][2 * (i4 % 2) + 1] = pu[1];
    };
    auto grad4 = [&](int kb, int i4) {      // dS, without the factor `scale`, which multiplies dK once at the end
      lf_elem4 dw;
#pragma unroll
      for (int e = 0; e < 4; ++e) dw[e] = lf_from_float(s[kb][4 * i4 + e] * dp[kb][4 * i4 + e]);
      const lf_u32x2 du = __builtin_bit_cast(lf_u32x2, dw);
      dsf[kb][i4 / 2][2 * (i4 % 2)] = du[0];
      dsf[kb][i4 / 2][2 * (i4 % 2) + 1] = du[1];
    };
    // per fragment: the read that is LF_BW_PF fragments ahead, and a direct load every other time
    auto ahead = [&](int i) {
      const int f = i + LF_BW_PF;
      fr[f] = f < NF ? frag(st, qb, f) : frag(st_n, qb_n, f - NF);
    };
    auto load = [&](int i) {
      if (loads && i % 2 == 0 && i / 2 < kLoads) issue(ld, i / 2);
      __builtin_amdgcn_sched_barrier(0);
    };
    // what is carried from block to block may have been moved between registers just now, by the vector ALU
#pragma unroll
    for (int f = 0; f < LF_BW_PF; ++f) asm volatile("" : "+v"(fr[f]));
    asm volatile(LF_BW_VALU_SETTLE : "+v"(fr[0]));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      ahead(i);
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        if (i == 0) lf_bw_mfma_zero(s[kb], fr[i], kf[kb][i]);
        else lf_bw_mfma_vvv(s[kb], fr[i], kf[kb][i]);
      }
      if (i == NS - 2) {
        dinit = read_stats(st, 1, qb);
        lse4[0] = read_stat4(st, 0, qb, 0);
#if LF_BW_VL
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) vl[0][kb] = v_lds[0][kb][tid];
#endif
      }
      load(i);
    }
#pragma unroll
    for (int ks = 0; ks < NS; ++ks) {
      ahead(NS + ks);
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
#if LF_BW_VL
        const lf_u32x4 vop = ks < LF_BW_VL ? vl[ks][kb] : vf[kb][ks - LF_BW_VL];
#else
        const lf_u32x4 vop = vf[kb][ks];
#endif
        if (ks == 0) lf_bw_mfma_from(dp[kb], fr[NS + ks], vop, dinit);
        else lf_bw_mfma_vvv(dp[kb], fr[NS + ks], vop);
#if LF_BW_VL
        if (ks + 1 < LF_BW_VL) vl[ks + 1][kb] = v_lds[ks + 1][kb][tid];
#endif
      }
      if (ks == 0) {
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) asm volatile(LF_BW_MFMA_DRAIN : "+v"(s[kb]));
      } else if (ks == 1) {
        LF_BW_HOLD(dinit);
      }
#pragma unroll
      for (int t = ks * 4 * KB / NS; t < (ks + 1) * 4 * KB / NS; ++t) {
        if (t % KB == 0 && t / KB < 3) lse4[t / KB + 1] = read_stat4(st, 0, qb, t / KB + 1);
        soft4(t % KB, t / KB);
      }
      load(NS + ks);
    }
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) asm volatile(LF_BW_VALU_SETTLE : "+v"(pf[kb][0]), "+v"(pf[kb][1]), "+v"(s[kb]));     // (s: P takes its place)
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      ahead(2 * NS + j);
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) lf_bw_mfma_hidden(dv[kb][j % LF_NDB], fr[2 * NS + j], pf[kb][j / LF_NDB]);
      if (j == 0) {
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) asm volatile(LF_BW_MFMA_DRAIN : "+v"(dp[kb]));
      }
#pragma unroll
      for (int t = j * 4 * KB / NT; t < (j + 1) * 4 * KB / NT; ++t) grad4(t % KB, t / KB);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) asm volatile(LF_BW_VALU_SETTLE : "+v"(dsf[kb][0]), "+v"(dsf[kb][1]));
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      ahead(2 * NS + NT + j);
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) lf_bw_mfma_hidden(dk[kb][j % LF_NDB], fr[2 * NS + NT + j], dsf[kb][j / LF_NDB]);
#if LF_BW_DS
      if (j % (NT / (2 * KB)) == 0) {
        const int t = j / (NT / (2 * KB)), kb = t / 2, half = t % 2, key = key0 + 32 * kb;
        bool store = true;
        if (masked) {
          store = key < p.Sk;
#if LF_MASK >= 1
          store = store && key <= q0;
#endif
#if LF_MASK == 2
          store = store && q0 - (min(key + 32, p.Sk) - 1) < p.window;
#endif
        }
        if (store) {
          ++ds_young;
          char* at = reinterpret_cast<char*>(ds_head) + 2048ll * (lf_bw_ds_row(q0 / 32, nkb, p.window) + key / 32);
          __builtin_nontemporal_store(dsf[kb][half], reinterpret_cast<lf_u32x4*>(at + 1024 * half + (half ? ds_off ^ 128u : ds_off)));
        }
      }
#endif
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int f = 0; f < LF_BW_PF; ++f) pre[f] = fr[NF + f];
  };
  // does the wave have a score to keep in queries q .. q + 31, and are all of them kept?
  auto need = [&](int q) {
    bool n = key0 < p.Sk && q < p.Sq;
#if LF_MASK >= 1
    n = n && q + 31 >= key0;
#endif
#if LF_MASK == 2
    n = n && q - klast < p.window;
#endif
    return n;
  };
  auto full = [&](int q) {
    bool n = key0 + 32 * KB <= p.Sk;
#if LF_MASK >= 1
    n = n && key0 + 32 * KB - 1 <= q;
#endif
#if LF_MASK == 2
    n = n && q + 31 - key0 < p.window;
#endif
    return n;
  };

  if (nsteps > 0) {
    aim();
#pragma unroll
    for (int j = 0; j < kLoads; ++j) issue(0, j);
    aim();
#pragma unroll
    for (int j = 0; j < kLoads; ++j) issue(1, j);
#if LF_BW_QSPLIT
    aim();
#pragma unroll
    for (int j = 0; j < kLoads; ++j) issue(2, j);
    LF_BW_BARRIER();
    read_ahead(0, 0);
    int st = 0, q0 = 64 * qt_begin + 32 * my_qb, left = ntq;
    // this wave's loads but the newest tile's, and stores of dS behind those, are done (the counter retires in order; waves
    // 0 and 1 have a load of statistics more); then every wave's
    auto stage = [&]() {
      asm volatile("" ::: "memory");
      if (wave < 2) lf_bw_wait<kLoads + 1, LF_BW_DS ? 2 * KB : 0>(ds_young);
      else lf_bw_wait<kLoads, LF_BW_DS ? 2 * KB : 0>(ds_young);
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      ds_young = 0;
    };
    for (int it = 0; it < nsteps; ++it) {
      const int st1 = (st + 1) & 3, st3 = (st + 3) & 3;
      stage();                    // the next tile has landed; every wave is done with the one before this
      aim();
      if (!need(q0)) {
#pragma unroll
        for (int j = 0; j < kLoads; ++j) issue(st3, j);
        read_ahead(st1, 0);
      } else if (full(q0)) {
        block(0, st, q0, false, true, st3, st1, 0);
      } else {
        block(0, st, q0, true, true, st3, st1, 0);
      }
      st = st1;
      q0 += 64;
      if (--left == 0) {
        left = ntq;
        q0 = 64 * qt_begin + 32 * my_qb;
#if LF_BW_DS
        ds_head += p.ds_sh;
#endif
      }
    }
#else
    LF_BW_BARRIER();
    read_ahead(0, 0);
    int st = 0, q0 = 64 * qt_begin, left = ntq;
    for (int it = 0; it < nsteps; ++it) {
      const int st1 = st == 2 ? 0 : st + 1, st2 = st == 0 ? 2 : st - 1;
      // (an instance each for the blocks that need the mask arithmetic and for those that do not: a branch per four
      // scores costs registers that are not there)
      if (!need(q0)) read_ahead(st, 1);
      else if (full(q0)) block(0, st, q0, false, false, 0, st, 1);
      else block(0, st, q0, true, false, 0, st, 1);
      // the next tile has landed; every wave is done with the one before this
#if LF_BW_DS
      // (stores of dS behind the loads stay in flight: the counter retires in order)
      asm volatile("" ::: "memory");
      if (ds_young == 4 * KB) __builtin_amdgcn_s_waitcnt(0x0070 | 4 * KB);
      else __builtin_amdgcn_s_waitcnt(0x0070);
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      ds_young = 0;
#else
      LF_BW_BARRIER();
#endif
      aim();
      if (!need(q0 + 32)) {
#pragma unroll
        for (int j = 0; j < kLoads; ++j) issue(st2, j);
        read_ahead(st1, 0);
      } else if (full(q0 + 32)) {
        block(1, st, q0 + 32, false, true, st2, st1, 0);
      } else {
        block(1, st, q0 + 32, true, true, st2, st1, 0);
      }
      st = st1;
      q0 += 64;
      if (--left == 0) {
        left = ntq;
        q0 = 64 * qt_begin;
#if LF_BW_DS
        ds_head += p.ds_sh;
#endif
      }
    }
#endif
    __builtin_amdgcn_s_waitcnt(0x0070);      // the last loads, against an empty range, before the LDS is given back
  }
#pragma unroll
  for (int kb = 0; kb < KB; ++kb)
#pragma unroll
    for (int db = 0; db < LF_NDB; ++db) asm volatile(LF_BW_MFMA_DRAIN_LAST : "+a"(dk[kb][db]), "+a"(dv[kb][db]));
#if LF_BW_QSPLIT
  // the sums of the waves that held the same keys, through LDS (nobody reads its tiles any more), lane by lane
  {
    lf_f32x4* sums = reinterpret_cast<lf_f32x4*>(&tiles[0][0][0]);
    static_assert(KB * LF_NDB * 8 * 128 * 16 <= (int)sizeof(tiles), "the sums fit the tiles");
    auto at = [&](int j, int i4) -> lf_f32x4& { return sums[(j * 4 + i4) * 128 + (tid & 127)]; };
    __syncthreads();
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int db = 0; db < LF_NDB; ++db)
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) {
          const int j = 2 * (kb * LF_NDB + db);
          if (my_qb == 1) {
            at(j, i4) = lf_f32x4{dk[kb][db][4 * i4], dk[kb][db][4 * i4 + 1], dk[kb][db][4 * i4 + 2], dk[kb][db][4 * i4 + 3]};
            at(j + 1, i4) = lf_f32x4{dv[kb][db][4 * i4], dv[kb][db][4 * i4 + 1], dv[kb][db][4 * i4 + 2], dv[kb][db][4 * i4 + 3]};
          }
        }
    __syncthreads();
    if (my_qb == 1) return;
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int db = 0; db < LF_NDB; ++db)
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) {
          const int j = 2 * (kb * LF_NDB + db);
          const lf_f32x4 x = at(j, i4), y = at(j + 1, i4);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            dk[kb][db][4 * i4 + e] += x[e];
            dv[kb][db][4 * i4 + e] += y[e];
          }
        }
  }
#endif
  // the parameters of the output are read only now: held over the loop they cost scalar registers it needs
  auto ep = (const LfAttnBwdParams __attribute__((address_space(4)))*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(ep));
  const float scale = ep->scale;
#if LF_BW_QSPLIT
  const unsigned rows_lds = lds0 + (unsigned)(KB * LF_NDB * 8 * 128 * 16 + wave * LF_BW_ROWS_LDS);      // behind the sums
  static_assert(KB * LF_NDB * 8 * 128 * 16 + kKeyWaves * LF_BW_ROWS_LDS <= (int)sizeof(tiles), "sums and rows fit the tiles");
#else
  static_assert(4 * LF_BW_ROWS_LDS <= (int)sizeof(tiles), "the rows fit the tiles");
  const unsigned rows_lds = lds0 + (unsigned)(wave * LF_BW_ROWS_LDS);
#if !LF_STAY
  __syncthreads();               // nobody reads the tiles any more
#endif
#endif
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
    const int first = key0 + 32 * kb;
#pragma unroll
    for (int db = 0; db < LF_NDB; ++db)
#pragma unroll
      for (int i = 0; i < 16; ++i) dk[kb][db][i] *= scale;
    lf_bw_store_rows(dk[kb], rows_lds, ep->dk + (long long)b * ep->dk_sb + (long long)hkv * ep->dk_sh + (long long)first * ep->dk_ss, ep->dk_ss,
                     p.Sk - first, lane);
    lf_bw_store_rows(dv[kb], rows_lds, ep->dv + (long long)b * ep->dv_sb + (long long)hkv * ep->dv_sh + (long long)first * ep->dv_ss, ep->dv_ss,
                     p.Sk - first, lane);
  }
}

#ifndef LF_BW_DQ_NT
#define LF_BW_DQ_NT 512  /* threads of lf_attn_bwd_dq, 32 query rows per wave */
#endif
#define LF_BW_DQ_PF 4    /* fragments read ahead of the MFMAs that take them */

#if LF_BW_DS
// dQ of LF_BW_DQ_NT / 2 query rows of one (batch, head), 32 per wave, from the dS that lf_attn_bwd_dkdv left: dQ^T += K^T dS^T.
// Bound by its loads: dS once, 2 bytes per visible score, and a K tile from L2 per 64 keys and workgroup, which return to a CU
// in order.  Causal bf16 B4 H32 S2048 D128, 545 MB of dS: 131 us (126 with the products left out; 152 where the loads of dS
// are plain ones and push K out of the L2), against 222 us of the kernel below, which forms dS again.  A step is 64 keys: the
// K tile, and every wave's own two blocks of dS, 4 KB in a row of memory; three LDS stages, one barrier.  Steps of 32 keys in
// 3 ... 6 stages: 143 ... 148 us.
extern "C" __global__ void __launch_bounds__(LF_BW_DQ_NT, LF_BW_DQ_NT / 256) lf_attn_bwd_dq(const LfAttnBwdParams p) {
  constexpr int kBM = LF_BW_DQ_NT / 2, kWaves = LF_BW_DQ_NT / 64, kS = 3;
  __shared__ __attribute__((aligned(256))) lf_elem k_tiles[kS][64 * LF_D];
  __shared__ __attribute__((aligned(256))) lf_elem ds_tiles[kS][kWaves][2 * 1024];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31;
  const int g = lane >> 5;

  const int nqt = (p.Sq + kBM - 1) / kBM;
  const int group = p.Hq / p.Hkv;
  int bhkv, row;
  if (!lf_slot_of_block(blockIdx.x, p.B * p.Hkv, group * nqt, LF_BW_GROUP, bhkv, row)) return;
  const int qt = nqt - 1 - row / group;
  const int hkv = bhkv % p.Hkv;
  const int b = bhkv / p.Hkv;
  const int h = hkv * group + row % group;
  const int q0 = kBM * qt;
  const int wq0 = q0 + 32 * wave;                    // first row of this wave

  int kt_begin = 0, kt_end = (p.Sk + 63) / 64;
  {
    const int qlast = min(q0 + kBM, p.Sq) - 1;
#if LF_MASK >= 1
    kt_end = min(kt_end, qlast / 64 + 1);
#endif
#if LF_MASK == 2
    const int lo = q0 - p.window + 1;
    if (lo > 0) kt_begin = lo / 64;
#endif
    (void)qlast;
  }
  const unsigned k_rowb = (unsigned)p.k_ss * 2u;
  const unsigned k_bytes = (unsigned)(((long long)(p.Sk - 1) * p.k_ss + LF_D) * 2);
  lf_u32x4 k_rs = lf_make_buffer(p.k + (long long)b * p.k_sb + (long long)hkv * p.k_sh, k_bytes);
  const unsigned k_loff = lf_bw_load_off(k_rowb, tid);
  // the wave's row of blocks; what it does not hold (keys behind the diagonal, past the last, in front of the window) lies
  // outside the range and arrives as zeros
  const int nkb = (p.Sk + 31) / 32, qb = wq0 / 32;
  const int row0 = lf_bw_ds_row(qb, nkb, p.window), row1 = lf_bw_ds_row(qb + 1, nkb, p.window);
  const int first = LF_MASK == 2 ? max(0, qb - (p.window + 30) / 32) : 0;      // its first key block
  const bool rows = wq0 < p.Sq;
  const lf_elem* ds_row = p.ds + ((long long)b * p.Hq + h) * p.ds_sh + 1024ll * (row0 + first);
#if LF_MASK == 2
  const int count = min(qb + 1, nkb) - first;
  (void)row1;
#else
  const int count = row1 - row0;
#endif
  lf_u32x4 ds_rs = lf_make_buffer(ds_row, rows && count > 0 ? 2048u * (unsigned)count : 0u);

  constexpr int kPasses = 64 * LF_CPR / LF_BW_DQ_NT;      // K loads of a wave per tile
  constexpr int kLoads = kPasses + 4;
  static_assert(kLoads * (kS - 2) < 16, "loads left in flight");
  const unsigned k0_lds = lf_lds_addr(k_tiles), ds0_lds = lf_lds_addr(ds_tiles);
  auto k_tile = [&](int st) { return k0_lds + (unsigned)(st * LF_BW_TILEB); };
  auto ds_tile = [&](int st) { return ds0_lds + (unsigned)((st * kWaves + wave) * 4096); };
  int ld_kt = kt_begin;
  auto issue = [&](int st) {
    if (ld_kt >= kt_end) k_rs[2] = ds_rs[2] = 0u;       // past the last tile: against an empty range
#pragma unroll
    for (int j = 0; j < 4; ++j)
      lf_dma_nt_to_lds_at(ds_rs, (unsigned)(2 * ld_kt - first) * 2048u + 1024u * (unsigned)j + 16u * (unsigned)lane,
                          ds_tile(st) + 1024u * (unsigned)j);
#pragma unroll
    for (int j = 0; j < kPasses; ++j) lf_bw_load_rows<LF_BW_DQ_NT>(k_rs, k_rowb, 64 * ld_kt, k_tile(st), k_loff, j, wave);
    ++ld_kt;
  };
  // does the wave have a score to keep in keys k .. k + 31 (lf_attn_bwd_dkdv has written those blocks)?
  auto need = [&](int k) {
    bool n = rows && k < p.Sk;
#if LF_MASK >= 1
    n = n && k <= wq0;
#endif
#if LF_MASK == 2
    n = n && min(k + 32, p.Sk) - 1 >= wq0 - p.window + 1;
#endif
    return n;
  };

  lf_f32x16 dq[LF_NDB];
#pragma unroll
  for (int db = 0; db < LF_NDB; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) dq[db][i] = 0.0f;
  const unsigned tr_off = lf_bw_tr_off(lane);
  // dS^T[key][query] fragments: lane % 32 the query, keys 16 * kk + 8 * half + 4 * g + 0 .. 3
  const int j16 = lane & 15, hq = (lane >> 4) & 1, u = 2 * hq + (j16 & 1);
  const unsigned ds_off = (unsigned)(512 * u + 64 * (g ^ u) + 16 * (j16 >> 2) + 8 * ((j16 >> 1) & 1));
  if (kt_begin < kt_end) {
#pragma unroll
    for (int s = 0; s < kS - 1; ++s) issue(s);
    int st = 0;
    for (int kt = kt_begin; kt < kt_end; ++kt) {
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_waitcnt((kLoads * (kS - 2)) | 0x70);          // the tile has landed (the next one's loads are in flight) ...
      __builtin_amdgcn_s_barrier();                       // ... for every wave, and every wave is done with the one before
      asm volatile("" ::: "memory");
      issue(st == 0 ? kS - 1 : st - 1);
      const unsigned kb0 = k_tile(st) + tr_off, sb0 = ds_tile(st) + ds_off;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        if (!need(64 * kt + 32 * kb)) continue;
#pragma unroll
        for (int kk = 2 * kb; kk < 2 * kb + 2; ++kk) {
          lf_u32x4 sf;
#pragma unroll
          for (int half = 0; half < 2; ++half) {
            const unsigned at = (half ? sb0 ^ 128u : sb0) + (unsigned)(2048 * kb + 256 * (kk & 1));
            const lf_u32x2 t = __builtin_bit_cast(lf_u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lf_bw_lds_s16x4)(size_t)at));
            sf[2 * half] = t[0];
            sf[2 * half + 1] = t[1];
          }
#pragma unroll
          for (int db = 0; db < LF_NDB; ++db)
            dq[db] = lf_mfma32(__builtin_bit_cast(lf_elem8, lf_bw_read_tr(kb0, 0, kk, db)), __builtin_bit_cast(lf_elem8, sf), dq[db]);
        }
      }
      st = st == kS - 1 ? 0 : st + 1;
    }
    __builtin_amdgcn_s_waitcnt(0x0070);      // the last loads, against an empty range, before the LDS is given back
  }
#pragma unroll
  for (int db = 0; db < LF_NDB; ++db) asm volatile(LF_BW_MFMA_DRAIN_LAST : "+a"(dq[db]));
#pragma unroll
  for (int db = 0; db < LF_NDB; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) dq[db][i] *= p.scale;
  static_assert(kWaves * LF_BW_ROWS_LDS <= (int)sizeof(ds_tiles), "the rows fit the tiles");
#if !LF_STAY
  __syncthreads();               // nobody reads the tiles any more
#endif
  lf_bw_store_rows(dq, ds0_lds + (unsigned)(wave * LF_BW_ROWS_LDS), p.dq + (long long)b * p.dq_sb + (long long)h * p.dq_sh + (long long)wq0 * p.dq_ss,
                   p.dq_ss, p.Sq - wq0, lane);
}
#else
// dQ of LF_BW_DQ_NT / 2 query rows of one (batch, head), 32 per wave.
// A wave walks blocks of 32 keys, two per 64-key tile, as lf_attn_bwd_dkdv walks blocks of queries: fragments through one
// read-ahead ring, three LDS stages, one barrier in the middle of a step.  Per block:
//   S^T = K Q^T
//   dP^T = V dO^T                    P between these MFMAs
//   dQ^T += K^T dS^T of the block before (it has no other product to hide dS behind); dS of this block between these
// What bounds it: an LDS fragment read (16 ... 24 cycles of the CU's LDS) per MFMA of a wave and the matrix work, with two
// waves per SIMD: 512 threads, or 256 with two workgroups per CU where their LDS fits (head dimension 64).  A wave's 256
// registers are dQ^T, Q^T and dO^T in 128 AGPRs and S^T, dP^T, two dS^T, fragments and addresses in 118 VGPRs.  Two row
// blocks per wave, half the LDS reads with one wave per SIMD, are slower (causal bf16 B4 H32 S2048 D128: 246 us): then
// nothing fills the gaps of a wave's own stream.  Against the form before (a copy of the K tile per read pattern, two
// stages, dS in front of its product; 4 waves per CU under a window or a softcap), us:
//   causal B4 H32 S2048 D128 223 -> 222, B2 32/8 S4096 378 -> 373, B2 16/8 S777 35 -> 25, B1 32/8 S2048 85 -> 71
//   the same with a softcap 383 -> 275; window 256 B4 32/8 S2048 151 -> 107, window 1024 259 -> 179
//   causal B8 16/4 S1000 D64 fp16 47 -> 42, B16 32/8 S300 48 -> 32
extern "C" __global__ void __launch_bounds__(LF_BW_DQ_NT, LF_BW_DQ_NT / 256) lf_attn_bwd_dq(const LfAttnBwdParams p) {
  constexpr int kBM = LF_BW_DQ_NT / 2;                           // query rows of a workgroup
  __shared__ __attribute__((aligned(256))) lf_elem tiles[3][2][64 * LF_D];        // K, V

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31;
  const int g = lane >> 5;

  const int nqt = (p.Sq + kBM - 1) / kBM;
  // As in lf_attn_bwd_dkdv: the q tiles of all query heads of a (batch, kv head) share its K / V tiles in one
  // XCD's L2, the long q tiles first.
  const int nrow = (p.Hq / p.Hkv) * nqt;                  // (query head of the group, q tile) per pair
  int bhkv, row;
  if (!lf_slot_of_block(blockIdx.x, p.B * p.Hkv, nrow, LF_BW_GROUP, bhkv, row)) return;
  const int qt = nqt - 1 - row / (p.Hq / p.Hkv);
  const int hkv = bhkv % p.Hkv;
  const int b = bhkv / p.Hkv;
  const int h = hkv * (p.Hq / p.Hkv) + row % (p.Hq / p.Hkv);
  const int q0 = kBM * qt;
  const int wq0 = q0 + 32 * wave;                    // first row of this wave
  const int nkt = (p.Sk + 63) / 64;

  // Q^T and dO^T of this lane's rows as B operands (d = 16*ks + 8*g .. +7)
  lf_u32x4 qf[LF_NKS], gf[LF_NKS];
  float delta_q;
  const int my_q = wq0 + l32, qr = min(my_q, p.Sq - 1);
  {
    const lf_elem* qrow = p.q + (long long)b * p.q_sb + (long long)h * p.q_sh + (long long)qr * p.q_ss;
    const lf_elem* grow = p.dout + (long long)b * p.do_sb + (long long)h * p.do_sh + (long long)qr * p.do_ss;
#pragma unroll
    for (int ks = 0; ks < LF_NKS; ++ks) {
      qf[ks] = *reinterpret_cast<const lf_u32x4*>(qrow + 16 * ks + 8 * g);
      gf[ks] = *reinterpret_cast<const lf_u32x4*>(grow + 16 * ks + 8 * g);
    }
#if LF_BW_DQ_NT == 256
    // delta of the row, half of its elements in each of two lanes: eight sums of LF_NKS products, then a tree, i.e. chains
    // as short as those of lf_attn_bwd_delta.  dO is in registers here anyway, so this costs a read of O, where a launch of
    // its own reads both.  Both launches against this one, us: causal B8 16/4 S1000 D64 52 / 43, B2 16/8 S777 D128 31 / 26,
    // B16 H8 S256 D128 20 / 16, unmasked B8 H16 S1024 D64 75 / 64.  The single workgroup that a CU holds of the larger
    // form has nothing to run beside these reads (causal B4 H32 S2048 D128 238 / 243): there delta has its launch.
    const lf_elem* orow = p.o + (long long)b * p.o_sb + (long long)h * p.o_sh + (long long)qr * p.o_ss;
    lf_u32x4 of[LF_NKS];
#pragma unroll
    for (int ks = 0; ks < LF_NKS; ++ks) of[ks] = *reinterpret_cast<const lf_u32x4*>(orow + 16 * ks + 8 * g);
    float t[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) t[e] = 0.0f;
#pragma unroll
    for (int ks = 0; ks < LF_NKS; ++ks) {
      const lf_elem8 ov = __builtin_bit_cast(lf_elem8, of[ks]), gv = __builtin_bit_cast(lf_elem8, gf[ks]);
#pragma unroll
      for (int e = 0; e < 8; ++e) t[e] += (float)ov[e] * (float)gv[e];
    }
    const float half = ((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7]));
    delta_q = half + __shfl_xor(half, 32, 64);
#endif
#pragma unroll
    for (int ks = 0; ks < LF_NKS; ++ks) asm volatile("" : "+a"(qf[ks]), "+a"(gf[ks]));
  }
  const long long ridx = ((long long)b * p.Hq + h) * p.Sq + qr;
  const float lse_q = my_q < p.Sq ? p.lse[ridx] : __builtin_inff();
#if LF_BW_DQ_NT == 256
  if (my_q < p.Sq && g == 0) p.delta[ridx] = -delta_q;     // for lf_attn_bwd_dkdv
#else
  delta_q = my_q < p.Sq ? -p.delta[ridx] : 0.0f;
#endif
#if LF_SOFTCAP
  const float sc_exp = p.scale / p.softcap * (2.0f * LF_LOG2E);   // 2^(s * sc_exp) = e^(2x)
  const float cexp = p.softcap * LF_LOG2E;                        // exponent of P: tanh x * cexp - L
#else
  const float cexp = p.scale * LF_LOG2E;
#endif

  lf_f32x16 dq[LF_NDB];
#pragma unroll
  for (int db = 0; db < LF_NDB; ++db) {
#pragma unroll
    for (int i = 0; i < 16; ++i) dq[db][i] = 0.0f;
    asm volatile("" : "+a"(dq[db]));
  }

  int kt_begin = 0, kt_end = nkt;
  {
    const int qlast = min(q0 + kBM, p.Sq) - 1;
#if LF_MASK >= 1
    kt_end = min(nkt, qlast / 64 + 1);
#endif
#if LF_MASK == 2
    const int lo = q0 - p.window + 1;
    if (lo > 0) kt_begin = lo / 64;
#endif
    (void)qlast;
  }
  const unsigned k_bytes = (unsigned)(((long long)(p.Sk - 1) * p.k_ss + LF_D) * 2);
  const unsigned v_bytes = (unsigned)(((long long)(p.Sk - 1) * p.v_ss + LF_D) * 2);
  lf_u32x4 k_rs = lf_make_buffer(p.k + (long long)b * p.k_sb + (long long)hkv * p.k_sh, k_bytes);
  lf_u32x4 v_rs = lf_make_buffer(p.v + (long long)b * p.v_sb + (long long)hkv * p.v_sh, v_bytes);
  const unsigned k_rowb = (unsigned)p.k_ss * 2u, v_rowb = (unsigned)p.v_ss * 2u;
  const unsigned k_loff = lf_bw_load_off(k_rowb, tid), v_loff = lf_bw_load_off(v_rowb, tid);
  constexpr int kPasses = 64 * LF_CPR / LF_BW_DQ_NT;      // loads of a wave per tile
  constexpr int kLoads = 2 * kPasses;
  const unsigned lds0 = lf_lds_addr(tiles);
  auto k_tile = [&](int st) { return lds0 + (unsigned)(2 * st * LF_BW_TILEB); };
  auto v_tile = [&](int st) { return lds0 + (unsigned)((2 * st + 1) * LF_BW_TILEB); };
  // the tile that is loaded next; past the last one the loads go out against an empty range
  int ld_kt = kt_begin - 1;
  auto aim = [&]() {
    if (++ld_kt >= kt_end) k_rs[2] = v_rs[2] = 0u;
  };
  auto issue = [&](int st, int j) {      // load j of kLoads
    if (j < kPasses) lf_bw_load_rows<LF_BW_DQ_NT>(k_rs, k_rowb, 64 * ld_kt, k_tile(st), k_loff, j, wave);
    else lf_bw_load_rows<LF_BW_DQ_NT>(v_rs, v_rowb, 64 * ld_kt, v_tile(st), v_loff, j - kPasses, wave);
  };

  unsigned rm_off = lf_bw_rm_off(l32, g), tr_off = lf_bw_tr_off(lane);
  asm volatile("" : "+v"(rm_off), "+v"(tr_off));
  constexpr int NS = LF_NKS, NT = 2 * LF_NDB, NF = 2 * NS + NT, PF = LF_BW_DQ_PF;      // fragments of a block
  static_assert(kLoads <= NS, "a block's loads go out during its first two phases");
  static_assert(PF <= NS, "the read-ahead of a block's first phase");
  // dS^T of the first / second block of a tile: B operands of the block after it
  lf_u32x4 ds[2][2];
#pragma unroll
  for (int kb = 0; kb < 2; ++kb) ds[kb][0] = ds[kb][1] = lf_u32x4{0u, 0u, 0u, 0u};
  constexpr unsigned kNone = ~0u;
  unsigned last = kNone;           // K rows in LDS of the block whose dS waits for its product
  auto frag_kt = [&](unsigned rows, int j) { return lf_bw_read_tr(rows + tr_off, 0, j / LF_NDB, j % LF_NDB); };
  // fragment i of block kb of the stage: K rows, V rows
  auto frag = [&](int st, int kb, int i) {
    if (i < NS) return lf_bw_read_rm(k_tile(st) + rm_off, 0, kb, i);
    return lf_bw_read_rm(k_tile(st) + rm_off, LF_BW_TILEB, kb, i - NS);
  };
  lf_u32x4 pre[PF];                // the next block's first fragments
  auto read_ahead = [&](int st, int kb) {
#pragma unroll
    for (int f = 0; f < PF; ++f) pre[f] = frag(st, kb, f);
  };
  // dQ of the last block before one that has nothing for this wave
  auto flush = [&](const int kb) {
    lf_u32x4 fr[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) fr[j] = frag_kt(last, j);
    asm volatile(LF_BW_VALU_SETTLE : "+v"(ds[kb][0]), "+v"(ds[kb][1]));
#pragma unroll
    for (int j = 0; j < NT; ++j)
      lf_bw_mfma_hidden(dq[j % LF_NDB], fr[j], ds[kb][j / LF_NDB]);
    last = kNone;
  };

  // One block of a wave: 32 keys (kb of stage st, first one k0) x its rows.  `loads`: those of stage `ld` are issued
  // between the MFMAs; the block read ahead is (st_n, kb_n).
  auto block = [&](const int kb, int st, int k0, const bool masked, const bool loads, int ld, int st_n, const int kb_n) {
    lf_u32x4 fr[NF + PF];
#pragma unroll
    for (int f = 0; f < PF; ++f) fr[f] = pre[f];
    lf_f32x16 s, dp;
    const unsigned own = k_tile(st) + (unsigned)(32 * kb * LF_BW_ROWB);
    // the first block of a wave adds zeros times its own keys (any other tile may hold no numbers yet)
    const unsigned before = last != kNone ? last : own;
    int rel = 0, room = 0;
    if (masked) {
      room = p.Sk - k0 - 4 * g;
      rel = my_q - k0 - 4 * g;            // query minus key of element 0
      asm volatile("" : "+v"(rel), "+v"(room));      // formed per block: what derives from them is not kept over the loop
    }
    // P of elements 4*i4 .. +3 in s (with a cap: times its derivative)
    auto soft4 = [&](int i4) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = 4 * i4 + e;
#if LF_SOFTCAP
        const float r = __builtin_amdgcn_rcpf(1.0f + lf_exp2(s[i] * sc_exp));     // 1 / (e^(2x) + 1), x = s * scale / cap
        float pv = lf_exp2((1.0f - 2.0f * r) * cexp - lse_q);
#else
        float pv = lf_exp2(s[i] * cexp - lse_q);
#endif
        if (masked) {
          pv = (8 * i4 + e < room && lf_bw_keep(rel - 8 * i4 - e, p.window)) ? pv : 0.0f;
        }
#if LF_SOFTCAP
        s[i] = pv * (4.0f * r * (1.0f - r));             // 1 - tanh^2
#else
        s[i] = pv;
#endif
      }
    };
    auto grad4 = [&](int i4) {      // dS, without the factor `scale`, which multiplies dQ once at the end
      lf_elem4 dw;
#pragma unroll
      for (int e = 0; e < 4; ++e) dw[e] = lf_from_float(s[4 * i4 + e] * (dp[4 * i4 + e] - delta_q));
      const lf_u32x2 du = __builtin_bit_cast(lf_u32x2, dw);
      ds[kb][i4 / 2][2 * (i4 % 2)] = du[0];
      ds[kb][i4 / 2][2 * (i4 % 2) + 1] = du[1];
    };
    // per fragment: the read that is PF fragments ahead, and a direct load every other time
    auto ahead = [&](int i) {
      const int f = i + PF;
      fr[f] = f < 2 * NS ? frag(st, kb, f) : f < NF ? frag_kt(before, f - 2 * NS) : frag(st_n, kb_n, f - NF);
    };
    auto load = [&](int i) {
      if (loads && i % 2 == 0 && i / 2 < kLoads) issue(ld, i / 2);
      __builtin_amdgcn_sched_barrier(0);
    };
    // what is carried from block to block may have been moved between registers just now, by the vector ALU
#pragma unroll
    for (int f = 0; f < PF; ++f) asm volatile("" : "+v"(fr[f]));
    asm volatile(LF_BW_VALU_SETTLE : "+v"(fr[0]));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      ahead(i);
      if (i == 0) lf_bw_mfma_first(s, fr[i], qf[i]);         // S^T[key][q]
      else lf_bw_mfma_vva(s, fr[i], qf[i]);
      load(i);
    }
#pragma unroll
    for (int ks = 0; ks < NS; ++ks) {
      ahead(NS + ks);
      if (ks == 0) lf_bw_mfma_first(dp, fr[NS + ks], gf[ks]);   // dP^T[key][q]
      else lf_bw_mfma_vva(dp, fr[NS + ks], gf[ks]);
      if (ks == 0) asm volatile(LF_BW_MFMA_DRAIN : "+v"(s));
#pragma unroll
      for (int t = ks * 4 / NS; t < (ks + 1) * 4 / NS; ++t) soft4(t);
      load(NS + ks);
    }
    asm volatile(LF_BW_VALU_SETTLE : "+v"(ds[kb ^ 1][0]), "+v"(ds[kb ^ 1][1]), "+v"(s));
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      ahead(2 * NS + j);
      lf_bw_mfma_hidden(dq[j % LF_NDB], fr[2 * NS + j], ds[kb ^ 1][j / LF_NDB]);
      if (j == 0) {
        asm volatile(LF_BW_MFMA_DRAIN : "+v"(dp));
      }
#pragma unroll
      for (int t = j * 4 / NT; t < (j + 1) * 4 / NT; ++t) grad4(t);
      __builtin_amdgcn_sched_barrier(0);
    }
    last = own;
#pragma unroll
    for (int f = 0; f < PF; ++f) pre[f] = fr[NF + f];
  };
  // does the wave have a score to keep in keys k .. k + 31, and are all of them kept?
  auto need = [&](int k) {
    bool n = wq0 < p.Sq && k < p.Sk;
#if LF_MASK >= 1
    n = n && k <= min(wq0 + 32, p.Sq) - 1;
#endif
#if LF_MASK == 2
    n = n && min(k + 32, p.Sk) - 1 >= wq0 - p.window + 1;
#endif
    return n;
  };
  auto full = [&](int k) {
    bool n = k + 31 < p.Sk;
#if LF_MASK >= 1
    n = n && k + 31 <= wq0;
#endif
#if LF_MASK == 2
    n = n && wq0 + 32 - 1 - k < p.window;
#endif
    return n;
  };

  if (kt_begin < kt_end) {
    aim();
#pragma unroll
    for (int j = 0; j < kLoads; ++j) issue(0, j);
    aim();
#pragma unroll
    for (int j = 0; j < kLoads; ++j) issue(1, j);
    LF_BW_BARRIER();
    read_ahead(0, 0);
    int st = 0;
    for (int kt = kt_begin; kt < kt_end; ++kt) {
      const int k0 = 64 * kt;
      const int st1 = st == 2 ? 0 : st + 1, st2 = st == 0 ? 2 : st - 1;
      if (!need(k0)) {
        if (last != kNone) flush(1);
        read_ahead(st, 1);
      } else if (full(k0)) {
        block(0, st, k0, false, false, 0, st, 1);
      } else {
        block(0, st, k0, true, false, 0, st, 1);
      }
      LF_BW_BARRIER();            // the next tile has landed; every wave is done with the one before this
      aim();
      if (!need(k0 + 32)) {
        if (last != kNone) flush(0);
#pragma unroll
        for (int j = 0; j < kLoads; ++j) issue(st2, j);
        read_ahead(st1, 0);
      } else if (full(k0 + 32)) {
        block(1, st, k0 + 32, false, true, st2, st1, 0);
      } else {
        block(1, st, k0 + 32, true, true, st2, st1, 0);
      }
      st = st1;
    }
    if (last != kNone) flush(1);
    __builtin_amdgcn_s_waitcnt(0x0070);      // the last loads, against an empty range, before the LDS is given back
  }
#pragma unroll
  for (int db = 0; db < LF_NDB; ++db) asm volatile(LF_BW_MFMA_DRAIN_LAST : "+a"(dq[db]));
#pragma unroll
  for (int db = 0; db < LF_NDB; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) dq[db][i] *= p.scale;
  static_assert(LF_BW_DQ_NT / 64 * LF_BW_ROWS_LDS <= (int)sizeof(tiles), "the rows fit the tiles");
#if !LF_STAY
  __syncthreads();               // nobody reads the tiles any more
#endif
  lf_bw_store_rows(dq, lds0 + (unsigned)(wave * LF_BW_ROWS_LDS), p.dq + (long long)b * p.dq_sb + (long long)h * p.dq_sh + (long long)wq0 * p.dq_ss,
                   p.dq_ss, p.Sq - wq0, lane);
}
#endif
