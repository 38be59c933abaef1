// lf_mask_bits.hip — a boolean mask as bits and tile classes, for lf_attn_prefill_swp -DLF_BIAS=2.
//
// A mask that reaches the framework as torch.bool (attn_mask of F.scaled_dot_product_attention, masked_fill, where) is read
// here once, a byte per element, and left as what the attention kernel can use without arithmetic:
//
//   words[unit][block of 32 rows][32 blocks of 32 keys] = {seen, hidden}   (p.part_acc, two 32-bit words)
//       bit t: some / not every element of the 32 x 32 block t is visible.  Dead is (0, 1), open (1, 0), mixed (1, 1).
//   bits[unit][block of 32 rows][block of 32 keys][16]                     (p.bias, 64-bit words; blocks that are not open)
//       word i: the lanes of a wave whose element i of S^T is visible.  Lane l, element i is row l % 32, key
//       8 * (i / 4) + 4 * (l / 32) + i % 4 of the block, as the accumulator holds it, so word i is the select of element i.
//
// unit = batch' * heads' + head', with batch' / head' collapsed to 0 where the mask is broadcast (p.bias_sb, p.bias_sh 0), one
// block of rows where one row is shared by all queries (p.bias_sq 0).  Rows past Sq repeat the last one, keys past Sk count as
// neither visible nor hidden (their bits are 0).
//
// p.obias = mask bytes [batch', head', Sq or 1, Sk] with byte strides p.ob_sb / ob_sh / ob_sq and key stride 1, p.rows = 1
// where True means visible and 0 where it means masked.  Grid (blocks of 32 rows, units, 1024 keys), 256 threads: a wave
// takes 32 rows x 256 keys.  Rows on 4-byte borders of a multiple of 4 keys: a lane holds 4 keys, its 32 four-byte loads (256
// consecutive bytes per load and wave) all in flight; any other alignment: one key per lane, byte loads, 64 keys at a time.
// What bounds it is the read of the mask and a launch's latency: [4, 1, 1536, 1536] 4.6 us, the form before, which wrote the
// 0 / -inf bias of mixed 128 x 64 blocks in 16 bits, 6.8.
//
// The reference has no counterpart: its mask ops are index predicates
// (loopfuse/torch_backend/ops.py:675-751) and a mask given as data is not skipped over.

extern "C" __global__ __launch_bounds__(256) void lf_mask_tiles(const LfAttnParams p) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nhh = p.bias_sh ? p.Hq : 1;
  const int nrb = gridDim.x, nkb = (p.Sk + 31) / 32, nwords = (p.Sk + 1023) / 1024;
  const int rb = blockIdx.x, chunk = blockIdx.z;
  const unsigned char* base = reinterpret_cast<const unsigned char*>(p.obias) + (long long)(blockIdx.y / nhh) * p.ob_sb +
                              (long long)(blockIdx.y % nhh) * p.ob_sh;
  const int q0 = 32 * rb;
  const int qlast = p.bias_sq ? p.Sq - 1 : 0;
  const int k0 = 1024 * chunk + 256 * wave;             // first key of the wave
  const long long at = (long long)blockIdx.y * nrb + rb;
  unsigned* bits = reinterpret_cast<unsigned*>(const_cast<lf_elem*>(p.bias)) + at * nkb * 32;
  __shared__ unsigned found[4][2];
  // key c of a block: where its 32 rows lie among the block's 32 words
  auto place = [](int c) { return 8 * (c >> 3) + 2 * (c & 3) + ((c >> 2) & 1); };
  unsigned seen = 0u, hidden = 0u;                       // bit t: of the wave's block t
  const unsigned long long align = reinterpret_cast<unsigned long long>(p.obias) | (unsigned long long)p.ob_sb |
                                   (unsigned long long)p.ob_sh | (unsigned long long)p.ob_sq | (unsigned long long)p.Sk;
  if (k0 >= p.Sk) {
    // nothing of the last chunk for this wave
  } else if ((align & 3) == 0) {
    const int j = k0 + 4 * lane;
    const bool in = j < p.Sk;                            // four keys are inside or outside together
    unsigned v[32];
#pragma unroll
    for (int r = 0; r < 32; ++r)
      v[r] = *reinterpret_cast<const unsigned*>(base + (long long)min(q0 + r, qlast) * p.ob_sq + (in ? j : k0));
    // byte e of rows8[b]: key e, bit u: row 8 * b + u
    unsigned rows8[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      rows8[b] = 0u;
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const unsigned x = v[8 * b + u];
        rows8[b] |= ((((x & 0x7f7f7f7fu) + 0x7f7f7f7fu) | x) & 0x80808080u) >> (7 - u);       // high bit of a byte: it is not zero
      }
      if (!p.rows) rows8[b] = ~rows8[b];
    }
    // bytes of four words -> words of four bytes
    const unsigned a0 = __builtin_amdgcn_perm(rows8[1], rows8[0], 0x05010400u), a1 = __builtin_amdgcn_perm(rows8[1], rows8[0], 0x07030602u);
    const unsigned b0 = __builtin_amdgcn_perm(rows8[3], rows8[2], 0x05010400u), b1 = __builtin_amdgcn_perm(rows8[3], rows8[2], 0x07030602u);
    unsigned w[4] = {__builtin_amdgcn_perm(b0, a0, 0x05040100u), __builtin_amdgcn_perm(b0, a0, 0x07060302u),
                     __builtin_amdgcn_perm(b1, a1, 0x05040100u), __builtin_amdgcn_perm(b1, a1, 0x07060302u)};
    const unsigned long long some = __builtin_amdgcn_ballot_w64(in && (w[0] | w[1] | w[2] | w[3]) != 0u);
    const unsigned long long less = __builtin_amdgcn_ballot_w64(in && (w[0] & w[1] & w[2] & w[3]) != ~0u);
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      seen |= (unsigned)((some >> (8 * t) & 0xffull) != 0ull) << t;
      hidden |= (unsigned)((less >> (8 * t) & 0xffull) != 0ull) << t;
    }
    if ((hidden >> (lane / 8)) & 1u) {
      unsigned* dst = bits + (long long)(k0 / 32 + lane / 8) * 32;
#pragma unroll
      for (int e = 0; e < 4; ++e) dst[place(4 * (lane & 7) + e)] = in ? w[e] : 0u;
    }
  } else {
#pragma unroll 1
    for (int it = 0; it < 4 && k0 + 64 * it < p.Sk; ++it) {
      const int j = k0 + 64 * it + lane;
      const bool in = j < p.Sk;
      unsigned char v[32];
#pragma unroll
      for (int r = 0; r < 32; ++r) v[r] = base[(long long)min(q0 + r, qlast) * p.ob_sq + (in ? j : k0)];
      unsigned w = 0u;
#pragma unroll
      for (int r = 0; r < 32; ++r) w |= (v[r] != 0 ? 1u : 0u) << r;
      if (!p.rows) w = ~w;
      const unsigned long long some = __builtin_amdgcn_ballot_w64(in && w != 0u), less = __builtin_amdgcn_ballot_w64(in && w != ~0u);
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        seen |= (unsigned)((unsigned)(some >> (32 * t)) != 0u) << (2 * it + t);
        hidden |= (unsigned)((unsigned)(less >> (32 * t)) != 0u) << (2 * it + t);
      }
      if ((hidden >> (2 * it + lane / 32)) & 1u)
        bits[(long long)(k0 / 32 + 2 * it + lane / 32) * 32 + place(lane & 31)] = in ? w : 0u;
    }
  }
  if (lane == 0) {
    found[wave][0] = seen;
    found[wave][1] = hidden;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    unsigned w = 0u;
#pragma unroll
    for (int u = 0; u < 4; ++u) w |= found[u][threadIdx.x] << (8 * u);
    reinterpret_cast<unsigned*>(p.part_acc)[2 * (at * nwords + chunk) + threadIdx.x] = w;
  }
}
