// lf_bias_classify.hip — tile classes of an additive score bias, or of a boolean mask, for lf_attn_prefill_swp -DLF_BIAS=1.
//
// Mask tensors reach the kernels as score biases of 0 / -inf (attn_mask of
// F.scaled_dot_product_attention, hand-written `scores + mask`, boolean masks turned into
// that form by the front end).  Most (q tile, kv tile) blocks of such a bias are all -inf
// (nothing of the block is visible: the attention kernel does not compute it, and does not
// walk it at either end of a q tile's range) or all zero (the block needs no bias at all);
// only the few blocks on the edge of the visible region mix values.  This kernel reads the
// bias once per distinct (batch, head) it holds and writes, per q tile (128 rows; 64 or 32 when the
// attention kernel packs query heads, which it does only for a bias shared by all heads) and kv
// tile of 64 keys,
//
//   class[unit][kv tile] = 0 dead | 1 zero | 2 mixed                (int32)
//
// into p.part_acc, unit = (batch' * heads' + head') * q_tiles + q_tile with batch' / head'
// collapsed to 0 where the bias is broadcast (stride 0).
// A dense bias of real numbers costs two loads per block: only blocks whose bottom-left and
// top-right corners are both masked, or both zero, are read in full.
//
// Grid (q tiles, batches' * heads', groups of 4 kv tiles), 256 threads: one wave per block,
// 32 eight-byte loads per lane, all in flight together.  Needs bias rows that start on 8-byte
// boundaries (p.bias_sq and the strides multiples of 4) and Sk >= 4.
//
// The reference has no counterpart: its mask ops are index predicates
// (loopfuse/torch_backend/ops.py:675-751) and a mask given as data is not skipped over.

#define LF_BC_BM LF_BM      /* rows of the attention kernel's q tile: 128, or 64 / 32 with packed query heads */
#define LF_BC_BN LF_BN

extern "C" __global__ __launch_bounds__(256) void lf_bias_classify(const LfAttnParams p) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nqt = (p.Sq + LF_BC_BM - 1) / LF_BC_BM;
  const int nkt = (p.Sk + LF_BC_BN - 1) / LF_BC_BN;
  const int nhh = p.bias_sh ? p.Hq : 1;
  const int qt = blockIdx.x;
  const int bb = blockIdx.y / nhh, hh = blockIdx.y % nhh;
  const int unit = (bb * nhh + hh) * nqt + qt;
  const int kt = 4 * blockIdx.z + wave;
  if (kt >= nkt) return;
  int* cls = reinterpret_cast<int*>(p.part_acc) + (long long)unit * nkt;
  const lf_elem* base = p.bias + (long long)bb * p.bias_sb + (long long)hh * p.bias_sh;
  const int q0 = qt * LF_BC_BM;
  const int qlast = min(q0 + LF_BC_BM, p.Sq) - 1;
  const int k0 = kt * LF_BC_BN;
  const int klast = min(k0 + LF_BC_BN, p.Sk) - 1;
  auto bits = [&](int q, int j) { return (unsigned)__builtin_bit_cast(unsigned short, base[(long long)q * p.bias_sq + j]); };
  auto is_zero = [](unsigned b16) { return (b16 & 0x7fffu) == 0u; };

  // candidates by two corners (wave-uniform values: every lane reads the same two elements)
  const unsigned bl = bits(qlast, k0), tr = bits(q0, klast);
  bool dead = lf_bias_masked(bl) && lf_bias_masked(tr);
  bool zero = is_zero(bl) && is_zero(tr);
  if (dead || zero) {
    // lane = (row in a group of 4, 4-key chunk): 8-byte loads, LF_BC_BM / 4 groups of 4 rows cover the tile
    const int j = k0 + 4 * (lane & 15), r4 = lane >> 4;
    const bool whole = j + 3 <= klast;
    const int jload = min(j, p.Sk - 4);        // the chunk that would run past Sk is read from Sk - 4 (and not used)
    // all loads of the lane go out before the first is looked at: one memory latency per block
    lf_u32x2 w[LF_BC_BM / 4];
#pragma unroll
    for (int u = 0; u < LF_BC_BM / 4; ++u) {
      const int q = min(q0 + 4 * u + r4, qlast);      // rows past the end re-read the last one
      w[u] = *reinterpret_cast<const lf_u32x2*>(base + (long long)q * p.bias_sq + jload);
    }
    if (whole) {
#pragma unroll
      for (int u = 0; u < LF_BC_BM / 4; ++u)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          dead = dead && lf_bias_masked2(w[u][e]);
          zero = zero && is_zero(w[u][e] & 0xffffu) && is_zero(w[u][e] >> 16);
        }
    } else if (j <= klast) {
      // the chunk that holds key Sk - 1: element by element
      for (int u = 0; u < LF_BC_BM / 4; ++u) {
        const int q = min(q0 + 4 * u + r4, qlast);
        for (int e = 0; j + e <= klast; ++e) {
          const unsigned b16 = bits(q, j + e);
          dead = dead && lf_bias_masked(b16);
          zero = zero && is_zero(b16);
        }
      }
    }
  }
  const bool all_dead = __builtin_amdgcn_ballot_w64(dead) == ~0ull;
  const bool all_zero = __builtin_amdgcn_ballot_w64(zero) == ~0ull;
  if (lane == 0) cls[kt] = all_dead ? 0 : (all_zero ? 1 : 2);
}

// Tile classes of a boolean mask, and its 0 / -inf form where the attention kernel reads it.
//
// A mask that reaches the framework as torch.bool used to be turned into a score bias by torch (two scalar fills,
// where, a fill and a copy for the padded rows) and was then read again by lf_bias_classify: six launches in which every
// element was written twice and read three times at two bytes each.  The attention kernel reads the bias of mixed
// blocks only, one to three per q tile of a causal or padding mask, so this kernel reads the bytes once, writes the
// classes as above and the bias of the mixed blocks; the rest of the bias buffer stays unwritten.
//
// p.obias = mask bytes [batch', head', Sq or 1, Sk] with byte strides p.ob_sb / ob_sh / ob_sq and key stride 1, p.rows = 1
// where True means visible and 0 where it means masked; p.bias = bias buffer, rows of a multiple of 8 elements on
// 16-byte borders (bias_sq = 0: one row shared by all queries, written by the first q tile).  Grid and blocks as above.
// Rows on 16-byte borders with whole 16-key pieces: 16 keys per lane, 16 rows per load, all loads of the block in
// flight together; any other alignment: one key per lane, 32 rows in flight.
// F.scaled_dot_product_attention with a [4, 1, 1536, 1536] mask, 32 heads, D 128, whole call: 137 -> 107 us, of which the
// attention kernel is 98.
__device__ __forceinline__ unsigned lf_mt_visible(unsigned w, unsigned flip) {
  // high bit of each byte: the byte is not zero (and then flipped where True means masked)
  return ((((w & 0x7f7f7f7fu) + 0x7f7f7f7fu) | w) & 0x80808080u) ^ flip;
}

__device__ __forceinline__ unsigned lf_mt_pair(unsigned vis, int sh) {
  // two keys, high bits of the bytes at bit sh and sh + 8 of vis -> 0 or -inf each
  constexpr unsigned kNegInf = LF_DTYPE == 0 ? 0xff80u : 0xfc00u;
  const unsigned lo = (vis >> (sh + 7)) & 1u, hi = (vis >> (sh + 15)) & 1u;
  return (lo ? 0u : kNegInf) | (hi ? 0u : kNegInf << 16);
}

extern "C" __global__ __launch_bounds__(256) void lf_mask_tiles(const LfAttnParams p) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nqt = (p.Sq + LF_BC_BM - 1) / LF_BC_BM;
  const int nkt = (p.Sk + LF_BC_BN - 1) / LF_BC_BN;
  const int nhh = p.bias_sh ? p.Hq : 1;
  const int qt = blockIdx.x;
  const int bb = blockIdx.y / nhh, hh = blockIdx.y % nhh;
  const int unit = (bb * nhh + hh) * nqt + qt;
  const int kt = 4 * blockIdx.z + wave;
  if (kt >= nkt) return;
  int* cls = reinterpret_cast<int*>(p.part_acc) + (long long)unit * nkt;
  const unsigned char* base = reinterpret_cast<const unsigned char*>(p.obias) + (long long)bb * p.ob_sb + (long long)hh * p.ob_sh;
  lf_elem* dst = const_cast<lf_elem*>(p.bias) + (long long)bb * p.bias_sb + (long long)hh * p.bias_sh;
  const bool shared = p.bias_sq == 0;                // one row for all queries
  const int q0 = qt * LF_BC_BM;
  const int qlast = shared ? q0 : min(q0 + LF_BC_BM, p.Sq) - 1;
  const int k0 = kt * LF_BC_BN;
  const unsigned flip = p.rows ? 0u : 0x80808080u;
  bool dead = true, zero = true;                     // over this lane's keys
  const unsigned long long align = reinterpret_cast<unsigned long long>(p.obias) | (unsigned long long)p.ob_sb |
                                   (unsigned long long)p.ob_sh | (unsigned long long)p.ob_sq | (unsigned long long)p.Sk;
  if ((align & 15) == 0) {
    const int j = k0 + 16 * (lane & 3), r16 = lane >> 2;
    const bool in = j < p.Sk;                        // Sk is a multiple of 16: a piece is inside or outside as a whole
    lf_u32x4 w[LF_BC_BM / 16];
#pragma unroll
    for (int u = 0; u < LF_BC_BM / 16; ++u)
      w[u] = *reinterpret_cast<const lf_u32x4*>(base + (long long)min(q0 + 16 * u + r16, qlast) * p.ob_sq + (in ? j : k0));
#pragma unroll
    for (int u = 0; u < LF_BC_BM / 16; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        w[u][e] = lf_mt_visible(w[u][e], flip);
        dead = dead && (!in || w[u][e] == 0u);
        zero = zero && (!in || w[u][e] == 0x80808080u);
      }
    const bool all_dead = __builtin_amdgcn_ballot_w64(dead) == ~0ull;
    const bool all_zero = __builtin_amdgcn_ballot_w64(zero) == ~0ull;
    if (lane == 0) cls[kt] = all_dead ? 0 : (all_zero ? 1 : 2);
    if (all_dead || all_zero || !in || (shared && qt != 0)) return;
#pragma unroll
    for (int u = 0; u < LF_BC_BM / 16; ++u) {
      const int q = q0 + 16 * u + r16;
      if (q > qlast) continue;
      lf_elem* row = dst + (long long)q * p.bias_sq + j;
#pragma unroll
      for (int h = 0; h < 2; ++h)
        *reinterpret_cast<lf_u32x4*>(row + 8 * h) = lf_u32x4{lf_mt_pair(w[u][2 * h], 0), lf_mt_pair(w[u][2 * h], 16),
                                                             lf_mt_pair(w[u][2 * h + 1], 0), lf_mt_pair(w[u][2 * h + 1], 16)};
    }
    return;
  }
  // one key per lane; 32 rows are read before the first is looked at, their bits kept for the store
  const int j = k0 + lane;
  const bool in = j < p.Sk;
  unsigned seen[LF_BC_BM / 32];
#pragma unroll
  for (int r0 = 0; r0 < LF_BC_BM; r0 += 32) {
    unsigned char v[32];
#pragma unroll
    for (int u = 0; u < 32; ++u) v[u] = base[(long long)min(q0 + r0 + u, qlast) * p.ob_sq + (in ? j : k0)];
    unsigned bits = 0u;
#pragma unroll
    for (int u = 0; u < 32; ++u) bits |= (v[u] != 0 ? 1u : 0u) << u;
    seen[r0 / 32] = p.rows ? bits : ~bits;
    dead = dead && (!in || seen[r0 / 32] == 0u);
    zero = zero && (!in || seen[r0 / 32] == ~0u);
  }
  const bool all_dead = __builtin_amdgcn_ballot_w64(dead) == ~0ull;
  const bool all_zero = __builtin_amdgcn_ballot_w64(zero) == ~0ull;
  if (lane == 0) cls[kt] = all_dead ? 0 : (all_zero ? 1 : 2);
  if (all_dead || all_zero || !in || (shared && qt != 0)) return;
#pragma unroll
  for (int r = 0; r < LF_BC_BM; ++r) {
    if (q0 + r > qlast) break;
    const unsigned short bits = (seen[r / 32] >> (r & 31)) & 1u ? 0 : (LF_DTYPE == 0 ? 0xff80 : 0xfc00);
    dst[(long long)(q0 + r) * p.bias_sq + j] = __builtin_bit_cast(lf_elem, bits);
  }
}
