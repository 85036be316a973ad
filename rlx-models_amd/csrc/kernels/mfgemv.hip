// Decode matmul of one to four activation rows on the matrix cores:
// y[m, n] = sum_k x[m, k] * dequant(W)[n, k] over packed weights
// (Op::DequantMatMul at decode sizes, crates/rlx-models-core/src/
// standard_decoder.rs:727-738).
//
// A lane owns two whole blocks of one weight row: lane (j, g) of a wave has
// blocks of row j, lane groups g = 0 .. 3 different ones.  Their codes go to
// the 16x16x32 MFMA as exact f16 integers, and the activations' operand row
// 4G + r holds row r's values in lane group G's positions and zeros
// elsewhere, so that result row 4G + r is row r's sum over the block of lane
// group G: it arrives in the registers of just the lanes that own the block,
// whose f32 scale it is multiplied by there.  Against dot products on the
// VALU the cost per weight does not grow with the rows (up to four); f32 rows
// are two f16 rows (hi, lo).
//
// Workgroups of eight waves walk tiles of 16 weight rows, the waves sharing a
// tile's K.  A 256-element unit of the 16 rows is read as row-contiguous
// 16-byte pieces, two or three units ahead, and laid into the wave's own LDS
// region, where the lanes pick their blocks up.  (Lanes reading their blocks
// straight from memory: 28 us where this takes 20.5, Q8_0 4096->24576; a
// scale per lane and 16 rows to a block, the usual operand: 23.4, 20.0 with
// Q4_1 against 16.6.)
//
// What bounds it: 8-bit codes the weights' bandwidth (Q8_0 4096->24576, one
// f32 row 31.9 -> 21.5 us, 5.0 TB/s; 12288->4096 19.6 -> 13.0); 4-bit ones the
// instructions per weight and the start (MLX, four bf16 rows 23.7 -> 17.7 us,
// 12288->4096 20.6 -> 13.1; Q4_K, four f32 rows 46.1 -> 19.5); small calls the
// activations' way to the first product (Q8_0 2048->2048 5.1 -> 4.3 us).  So
// each wave prepares the activations of its own units, without a barrier, and
// asks for them ahead of the weights (12288->4096, MLX, four bf16 rows: 16.6
// us with the workgroup's maxima and the weights first, 15.2 by wave, 13.1
// with the activations first).
#include "common.hip.h"
#include "f16dq.hip.h"
#include "gemv_args.h"

namespace rlxq {

template <int SCH> constexpr int mf_order() {
  return SCH == SCH_MLX4 ? 2 : SCH == SCH_Q4_1 ? 1 : 0;
}
template <int SCH> constexpr bool mf_has_m() { return SCH == SCH_Q4_1 || SCH == SCH_Q4_K || SCH == SCH_MLX4; }
// Bytes of a row per unit (256 elements).
template <int SCH> constexpr int mf_seg() {
  return SCH == SCH_Q4_1 ? 160 : SCH == SCH_Q8_0 ? 272 : SCH == SCH_Q4_K ? 144 : SCH == SCH_MLX4 ? 128 : 208;
}
// Bytes between rows in LDS: an odd number of 16-byte pieces.
template <int SCH> constexpr int mf_lrow() {
  return SCH == SCH_Q4_1 ? 176 : SCH == SCH_Q8_0 ? 272 : SCH == SCH_Q4_K || SCH == SCH_MLX4 ? 144 : 240;
}

// What lane (j, g) loads of row j's unit: its two blocks.  Q4_1, Q8_0, MLX:
// blocks 2g and 2g + 1 (40, 68, 32 bytes; MLX: and their scales and biases).
// Q4_K: the 32 bytes whose low and high nibbles are those blocks, and the
// super-block's header.  Q6_K: the 32 ql bytes holding blocks 4n + i and 4n +
// i + 2 (n = g / 2, i = g % 2), the 32 qh bytes with their top bits, the
// blocks' scale bytes and d.
template <int SCH>
struct MfRaw {
  uint32_t c[SCH == SCH_Q4_1 ? 10 : SCH == SCH_Q8_0 ? 17 : SCH == SCH_Q6_K ? 16 : 8];
  uint32_t h[4];
};

RLXQ_DEV uint32_t mf_u32(const uint8_t* p) { return *reinterpret_cast<const uint32_t*>(p); }

// Reads the lane's two blocks from its row's region rp (off: 0 or 2, the
// super-block's first byte in it, Q6_K).
template <int SCH>
RLXQ_DEV void mf_read(const uint8_t* rp, int g, uint32_t off, MfRaw<SCH>& r) {
  auto v4 = [](const uint8_t* p, uint32_t* o) {
    const u32x4_t v = *reinterpret_cast<const u32x4_t*>(p);
#pragma unroll
    for (int e = 0; e < 4; e++) o[e] = v[e];
  };
  if constexpr (SCH == SCH_Q4_1) {
#pragma unroll
    for (int q = 0; q < 5; q++) {
      const uint2 v = *reinterpret_cast<const uint2*>(rp + 40 * g + 8 * q);
      r.c[2 * q] = v.x;
      r.c[2 * q + 1] = v.y;
    }
  } else if constexpr (SCH == SCH_Q8_0) {
#pragma unroll
    for (int q = 0; q < 17; q++) r.c[q] = mf_u32(rp + 68 * g + 4 * q);
  } else if constexpr (SCH == SCH_Q4_K) {
    v4(rp, r.h);
    v4(rp + 16 + 32 * g, r.c);
    v4(rp + 32 + 32 * g, r.c + 4);
  } else if constexpr (SCH == SCH_MLX4) {
    v4(rp + 32 * g, r.c);
    v4(rp + 32 * g + 16, r.c + 4);
  } else {
    uint32_t l[9], q[9];
#pragma unroll
    for (int e = 0; e < 9; e++) {
      l[e] = mf_u32(rp + 32 * g + 4 * e);
      q[e] = mf_u32(rp + 128 + 32 * (g >> 1) + 4 * e);
    }
#pragma unroll
    for (int e = 0; e < 8; e++) {
      r.c[e] = align_bytes(l[e + 1], l[e], off);
      // (the qh bits of the lane's first block to the bottom)
      r.c[8 + e] = align_bytes(q[e + 1], q[e], off) >> (2 * (g & 1));
    }
    const uint8_t* sp = rp + 192 + 8 * (g >> 1) + off + 2 * (g & 1);
    r.h[0] = *reinterpret_cast<const uint16_t*>(sp);
    r.h[1] = *reinterpret_cast<const uint16_t*>(sp + 4);
    r.h[2] = *reinterpret_cast<const uint16_t*>(rp + 208 + off);
  }
}

// Lane exchanges on the VALU: v of lane ^ 1 and ^ 2 (quad permutations), and
// sums with lanes ^ 16, ^ 32.
template <int ctrl>
RLXQ_DEV float mf_dpp(float v) {
  return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v), ctrl, 0xf, 0xf, true));
}
template <class F>
RLXQ_DEV float mf_rows(float v, F f) {
  typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
  u32x2_t p = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false));
  v = f(__uint_as_float(p.x), __uint_as_float(p.y));
  p = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false));
  return f(__uint_as_float(p.x), __uint_as_float(p.y));
}

// The four MFMA operands of block i (0, 1) of the lane: 8 codes each as exact
// f16 (1024 + code by bit pattern, then the offset).
template <int SCH, int i, int e>
RLXQ_DEV f16x8_t mf_codes(const MfRaw<SCH>& r) {
  uint32_t u0, u1;
  if constexpr (SCH == SCH_Q4_1 || SCH == SCH_MLX4) {
    const uint32_t c = SCH == SCH_Q4_1 ? r.c[5 * i + 1 + e] : r.c[4 * i + e];
    u0 = c & 0x0F0F0F0Fu;
    u1 = (c >> 4) & 0x0F0F0F0Fu;
  } else if constexpr (SCH == SCH_Q4_K) {
    u0 = (r.c[2 * e] >> (4 * i)) & 0x0F0F0F0Fu;
    u1 = (r.c[2 * e + 1] >> (4 * i)) & 0x0F0F0F0Fu;
  } else if constexpr (SCH == SCH_Q8_0) {
    u0 = (i ? r.c[9 + 2 * e] : align_bytes(r.c[2 * e + 1], r.c[2 * e], 2)) ^ 0x80808080u;
    u1 = (i ? r.c[10 + 2 * e] : align_bytes(r.c[2 * e + 2], r.c[2 * e + 1], 2)) ^ 0x80808080u;
  } else {
    static_assert(SCH == SCH_Q6_K, "format");
    // code (0..63) + 96 per byte, so that code - 32 = byte - 128 (the qh
    // dwords come shifted to the lane's first block)
    u0 = (((r.c[2 * e] >> (4 * i)) & 0x0F0F0F0Fu) | (i ? r.c[8 + 2 * e] & 0x30303030u : (r.c[8 + 2 * e] << 4) & 0x30303030u)) + 0x60606060u;
    u1 = (((r.c[2 * e + 1] >> (4 * i)) & 0x0F0F0F0Fu) | (i ? r.c[9 + 2 * e] & 0x30303030u : (r.c[9 + 2 * e] << 4) & 0x30303030u)) + 0x60606060u;
  }
  const _Float16 off = (SCH == SCH_Q8_0 || SCH == SCH_Q6_K) ? (_Float16)-1152.f : (_Float16)-1024.f;
  const f16x2_t of = {off, off};
  const f16x2_t w[4] = {magic_lo(u0) + of, magic_hi(u0) + of, magic_lo(u1) + of, magic_hi(u1) + of};
  return f16x8_t{w[0].x, w[0].y, w[1].x, w[1].y, w[2].x, w[2].y, w[3].x, w[3].y};
}

// A block's record in LDS: the inverse of each row's scale, a power of two,
// and for formats with a min / bias each row's sum.  One and two rows: MR (2
// MR) f32; four: the exponents as the bytes of a dword, and the sums in an
// array of their own behind those (four f32 rows then still fit the LDS at K =
// 8192).
template <int MR, bool HM> constexpr int mf_rec() { return MR == 4 ? 1 : HM ? 2 * MR : MR; }   // dwords
template <int MR, bool HM>
RLXQ_DEV void mf_record(const uint32_t* recs, const float* sums, int blk, float (&inv)[MR], float (&sum)[MR]) {
  const uint32_t* p = recs + blk * mf_rec<MR, HM>();
  if constexpr (MR == 4) {
    const uint32_t e = *p;
#pragma unroll
    for (int r = 0; r < 4; r++) inv[r] = __uint_as_float((r < 3 ? e << (23 - 8 * r) : e >> 1) & 0x7f800000u);
    if constexpr (HM) {
      const f32x4_t v = *reinterpret_cast<const f32x4_t*>(sums + 4 * blk);
#pragma unroll
      for (int r = 0; r < 4; r++) sum[r] = v[r];
    }
  } else if constexpr (mf_rec<MR, HM>() == 1) {
    inv[0] = __uint_as_float(*p);
  } else if constexpr (mf_rec<MR, HM>() == 2) {
    const uint2 v = *reinterpret_cast<const uint2*>(p);
    inv[0] = __uint_as_float(v.x);
    (HM ? sum[0] : inv[MR - 1]) = __uint_as_float(v.y);
  } else {
    const u32x4_t v = *reinterpret_cast<const u32x4_t*>(p);
    inv[0] = __uint_as_float(v[0]);
    inv[1] = __uint_as_float(v[1]);
    sum[0] = __uint_as_float(v[2]);
    sum[1] = __uint_as_float(v[3]);
  }
}

// LDS: x fragments [K / 32][4][MS NH] of 16 bytes, 8 * 4 * MS NH zero
// fragments' worth, the blocks' records, partial sums [2][8 waves][64] f32,
// then the waves' weight regions.
template <int SCH, bool XBF, int MR, int D>
RLXQ_DEV void mf_body(const rlxq_gemv_args& a) {
  constexpr int W = 8;
  // f32 rows are f16 hi and lo: as rows of their own up to two, as two
  // products into the same sums past that
  constexpr int NH = !XBF && MR > 2 ? 2 : 1, MS = XBF || MR > 2 ? MR : 2 * MR, FS = MS * NH;
  constexpr int SEG = mf_seg<SCH>(), PPR = SEG / 16, LROW = mf_lrow<SCH>(), ORD = mf_order<SCH>();
  constexpr int NP = 16 * PPR, NL = (NP + 63) / 64;
  constexpr bool HM = mf_has_m<SCH>(), MLX = SCH == SCH_MLX4, Q6 = SCH == SCH_Q6_K;
  constexpr int RF = mf_rec<MR, HM>();
  extern __shared__ __align__(16) uint8_t mf_lds[];
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 15, g = lane >> 4;
  const int K = a.K, nu = K / 256, nblk = K / 32;
  uint8_t* xs = mf_lds;
  uint8_t* zs = xs + nblk * 64 * FS;
  uint32_t* recs = reinterpret_cast<uint32_t*>(zs + 8 * 64 * FS);
  float* sums = reinterpret_cast<float*>(recs + nblk * RF);
  float* red = sums + (MR == 4 && HM ? 4 * nblk : 0);
  uint8_t* reg = reinterpret_cast<uint8_t*>(red + 2 * W * 64) + wv * (16 * LROW);

  // the wave's units of every tile of 16 weight rows (the last tile ends with
  // row N - 1 and shares rows with the one before it: the same sums, written
  // twice)
  const int u0 = wv * nu / W, cnt = (wv + 1) * nu / W - u0;
  const int ntile = (int)((a.N + 15) / 16), ntw = (ntile - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x;
  const int total = ntw * cnt;
  auto tile_row = [&](int t) { return (int64_t)t * 16 + 16 <= a.N ? (int64_t)t * 16 : a.N - 16; };

  // weight pieces of a unit, in row order: piece p is 16-byte unit p % PPR of
  // row p / PPR (lanes past the last repeat it)
  uint32_t src[NL];
  int dst[NL];
#pragma unroll
  for (int q = 0; q < NL; q++) {
    const int p = lane + 64 * q < NP ? lane + 64 * q : NP - 1;
    src[q] = (uint32_t)((p / PPR) * a.rb) + (p % PPR) * 16;
    dst[q] = (p / PPR) * LROW + (p % PPR) * 16;
  }
  u32x4_t wr[D][NL];
  uint32_t hr[D][MLX ? 4 : 1];   // MLX: scales and biases of the lane's blocks; Q6_K: row j's last dword
  const uint32_t tsrc = (uint32_t)(j * a.rb);
  const int gsh = MLX ? 31 - __builtin_clz((unsigned)a.group / 32u) : 0;   // blocks per group, as a shift
  const uint32_t srow = MLX ? (uint32_t)(j * (nblk >> gsh)) : 0u;
  int lt = blockIdx.x, lu = 0, li = 0;   // the next load's tile and unit
  auto load = [&](auto Q) {
    if (li >= total) return;
    li++;
    const int64_t n0 = tile_row(lt);
    const int u = u0 + lu;
    const uint8_t* wb = a.w + n0 * a.rb + (int64_t)u * (Q6 ? 210 : SEG);
    if constexpr (Q6) {
      // 210-byte super-blocks at 2-byte alignment, read from the dword they
      // start in (13 pieces and a last dword; nothing past the super-block and
      // the two bytes before it.  Rows are whole dwords.)
      const uint32_t off = (uint32_t)reinterpret_cast<uintptr_t>(wb) & 2u;
      wb -= off;
      const uint16_t* p = reinterpret_cast<const uint16_t*>(wb + tsrc + 208);
      hr[Q.value][0] = (uint32_t)p[0] | ((uint32_t)p[off >> 1] << 16);
    }
#pragma unroll
    for (int q = 0; q < NL; q++) {
      const uint4 v = ld_u128(wb + src[q]);
      wr[Q.value][q] = u32x4_t{v.x, v.y, v.z, v.w};
    }
    if constexpr (MLX) {
      const int64_t s0 = n0 * (nblk >> gsh);
      const uint32_t gi = srow + (uint32_t)((8 * u + 2 * g) >> gsh);
      const uint16_t* s16 = reinterpret_cast<const uint16_t*>(a.scales) + s0 + gi;
      const uint16_t* b16 = reinterpret_cast<const uint16_t*>(a.biases) + s0 + gi;
      const uint32_t* s32 = reinterpret_cast<const uint32_t*>(a.scales) + s0 + gi;
      const uint32_t* b32 = reinterpret_cast<const uint32_t*>(a.biases) + s0 + gi;
      hr[Q.value][0] = a.sb_bf16 ? (uint32_t)s16[0] : s32[0];
      hr[Q.value][2] = a.sb_bf16 ? (uint32_t)b16[0] : b32[0];
      if (gsh == 0) {   // (groups of 32: the second block's are the next ones)
        hr[Q.value][1] = a.sb_bf16 ? (uint32_t)s16[1] : s32[1];
        hr[Q.value][3] = a.sb_bf16 ? (uint32_t)b16[1] : b32[1];
      }
    }
    if (++lu == cnt) lu = 0, lt += gridDim.x;
  };

  // The activation rows over the wave's own units as f16 fragments, each
  // block of 32 scaled by the power of two that puts its maximum in [2^14,
  // 2^15): what a block keeps does not depend on the others', and within it an
  // element loses bits only 2^-17 below the maximum (f32, of 22) or 2^-31
  // (bf16).  (One power of two for a wave's whole stretch: what lies 2^-24
  // below its largest element kept ten bits, though that element may meet
  // zero weights alone.  The scale per block costs Q6_K 3 to 5%, 4096->24576
  // with one f32 row 23.8 -> 24.6 us, and the others up to 2%.)  Piece p: positions 8 (p % 4) .. of block p / 4 in
  // code order (natural, GGUF nibbles, MLX nibbles); a block's four pieces are
  // four neighbouring lanes.  A wave reads only what it wrote: no barrier
  // before the first tile's end.
  const int p0 = u0 * 32, p1 = (u0 + cnt) * 32;
  struct Piece { uint32_t w[XBF ? 4 : 8]; };   // as read (bf16 pairs or f32)
  auto ldx = [&](int row, int p) {
    const int i = p & 3;
    const int64_t e0 = (int64_t)(row < a.M ? row : a.M - 1) * K + (p >> 2) * 32 + (ORD == 1 ? 4 * i : 8 * i);
    const int64_t e1 = e0 + (ORD == 1 ? 16 : 4);
    Piece v;
    if constexpr (XBF) {
      const uint16_t* x = reinterpret_cast<const uint16_t*>(a.x);
      const uint2 c0 = *reinterpret_cast<const uint2*>(x + e0), c1 = *reinterpret_cast<const uint2*>(x + e1);
      v.w[0] = c0.x; v.w[1] = c0.y; v.w[2] = c1.x; v.w[3] = c1.y;
    } else {
      const uint32_t* x = reinterpret_cast<const uint32_t*>(a.x);
      const uint4 c0 = *reinterpret_cast<const uint4*>(x + e0), c1 = *reinterpret_cast<const uint4*>(x + e1);
      v.w[0] = c0.x; v.w[1] = c0.y; v.w[2] = c0.z; v.w[3] = c0.w;
      v.w[4] = c1.x; v.w[5] = c1.y; v.w[6] = c1.z; v.w[7] = c1.w;
    }
    return v;
  };
  {
    // Each lane's first NV pieces of a row are asked for ahead of the weights:
    // loads return in order.
    constexpr int NV = XBF || MR <= 2 ? 3 : 1;
    Piece v0[NV][MR];
#pragma unroll
    for (int q = 0; q < NV; q++)
      if (p0 + 64 * q < p1) {
        const int p = p0 + 64 * q + lane < p1 ? p0 + 64 * q + lane : p1 - 1;
#pragma unroll
        for (int r = 0; r < MR; r++) v0[q][r] = ldx(r, p);
      }
    static_for<D>([&](auto Q) { load(Q); });
    for (int p = lane; p < 8 * 4 * FS; p += 64) *reinterpret_cast<u32x4_t*>(zs + 16 * p) = u32x4_t{0u, 0u, 0u, 0u};
    auto put = [&](int r, int p, const Piece& v) {
      float mx = 0.f;
      if constexpr (XBF) {
        // (as integers: a NaN's bits are above every number's)
        typedef uint16_t u16x2_t __attribute__((ext_vector_type(2)));
        u16x2_t mh = {0, 0};
#pragma unroll
        for (int e = 0; e < 4; e++)
          mh = __builtin_elementwise_max(mh, __builtin_bit_cast(u16x2_t, v.w[e] & 0x7fff7fffu));
        const uint32_t h = mh.x > mh.y ? mh.x : mh.y;
        mx = __uint_as_float(h > 0x7f80u ? 0x7f800000u : h << 16);
      } else {
#pragma unroll
        for (int e = 0; e < 8; e++) mx = fmaxf(mx, fabsf(__uint_as_float(v.w[e])));
      }
      mx = fmaxf(mx, mf_dpp<0xB1>(mx));
      mx = fmaxf(mx, mf_dpp<0x4E>(mx));
      // (by exponent; a block that is not finite stays as it is)
      const uint32_t ex = __float_as_uint(mx) >> 23;
      int sh = 141 - (int)ex;
      sh = ex >= 255u ? 0 : (sh > 126 ? 126 : sh);
      const float s = __uint_as_float((uint32_t)(127 + sh) << 23), inv = __uint_as_float((uint32_t)(127 - sh) << 23);
      uint32_t hi[4], lo[4];
      float th = 0.f, tl = 0.f;
      const f16x2_t one = {(_Float16)1.f, (_Float16)1.f};
      float w[8];
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const int q = ORD == 2 ? (e < 4 ? 2 * e : 2 * (e - 4) + 1) : e;
        if constexpr (XBF) w[e] = __uint_as_float(q & 1 ? v.w[q / 2] & 0xffff0000u : v.w[q / 2] << 16) * s;
        else w[e] = __uint_as_float(v.w[q]) * s;
      }
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const uint32_t h0 = f32_to_f16_bits(w[2 * e]), h1 = f32_to_f16_bits(w[2 * e + 1]);
        hi[e] = h0 | (h1 << 16);
        if constexpr (HM) th = __builtin_amdgcn_fdot2(as_h2(hi[e]), one, th, false);
        if constexpr (!XBF) {
          // (the remainder is exact in f32; rounded once more)
          const uint32_t l0 = f32_to_f16_bits(w[2 * e] - f16_bits_to_f32(h0));
          const uint32_t l1 = f32_to_f16_bits(w[2 * e + 1] - f16_bits_to_f32(h1));
          lo[e] = l0 | (l1 << 16);
          if constexpr (HM) tl = __builtin_amdgcn_fdot2(as_h2(lo[e]), one, tl, false);
        }
      }
      *reinterpret_cast<u32x4_t*>(xs + (p * FS + r) * 16) = u32x4_t{hi[0], hi[1], hi[2], hi[3]};
      if constexpr (!XBF) *reinterpret_cast<u32x4_t*>(xs + (p * FS + MR + r) * 16) = u32x4_t{lo[0], lo[1], lo[2], lo[3]};
      // (all four lanes of a block store its record)
      const int blk = p >> 2;
      if constexpr (MR == 4) reinterpret_cast<uint8_t*>(recs + blk)[r] = (uint8_t)(127 - sh);
      else recs[blk * RF + r] = __float_as_uint(inv);
      if constexpr (HM) {
        float t = th + tl;
        t += mf_dpp<0xB1>(t);
        t += mf_dpp<0x4E>(t);
        if constexpr (MR == 4) sums[4 * blk + r] = t * inv;
        else recs[blk * RF + MR + r] = __float_as_uint(t * inv);
      }
    };
#pragma unroll
    for (int q = 0; q < NV; q++)
      if (p0 + 64 * q + lane < p1) {
#pragma unroll
        for (int r = 0; r < MR; r++) put(r, p0 + 64 * q + lane, v0[q][r]);
      }
    for (int p = p0 + 64 * NV + lane; p < p1; p += 64)
#pragma unroll
      for (int r = 0; r < MR; r++) put(r, p, ldx(r, p));
    // (the lanes' reads below cross lanes: not before these stores, some of
    // which are conditional)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }

  // The lane's x operand: row 4G + r of an MFMA's 16 takes row r's values of
  // the blocks of lane group G, so only the lanes with G == g hold any; the
  // others read zeros.
  const bool xlive = (j >> 2) == g;
  const uint8_t* xp = xlive ? xs + ((2 * g) * 4 * FS + (j & 3) % MS) * 16 : zs;
  const int xstep = xlive ? 8 * 64 * FS : 0;
  // (Q6_K: blocks 4n + i and 4n + i + 2)
  constexpr int B1 = Q6 ? 2 : 1;
  if constexpr (Q6) xp = xlive ? xs + ((4 * (g >> 1) + (g & 1)) * 4 * FS + (j & 3) % MS) * 16 : zs;
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  float acc[MS];
#pragma unroll
  for (int r = 0; r < MS; r++) acc[r] = 0.f;
  int ct = blockIdx.x, cu = 0, buf = 0, turn = 0;
  for (int i = 0; i < total; i += D) {
    static_for<D>([&](auto Q) {
      if (i + Q.value >= total) return;
      const int u = u0 + cu;
      // the wave's region is its own: its stores and reads are ordered by the
      // wave's in-order LDS queue (every lane stores, so that no lane's read
      // can be moved before another's store)
#pragma unroll
      for (int q = 0; q < NL; q++) *reinterpret_cast<u32x4_t*>(reg + dst[q]) = wr[Q.value][q];
      uint32_t off = 0;
      if constexpr (Q6) {
        *reinterpret_cast<uint32_t*>(reg + j * LROW + 208) = hr[Q.value][0];
        off = (uint32_t)(reinterpret_cast<uintptr_t>(a.w) + (uint32_t)u * 210) & 2u;
      }
      asm volatile("" ::: "memory");
      MfRaw<SCH> r;
      mf_read<SCH>(reg + j * LROW, g, off, r);
      if constexpr (MLX) {
        r.h[0] = hr[Q.value][0];
        r.h[2] = hr[Q.value][2];
        r.h[1] = gsh == 0 ? hr[Q.value][1] : r.h[0];
        r.h[3] = gsh == 0 ? hr[Q.value][3] : r.h[2];
      }
      asm volatile("" ::: "memory");
      load(Q);
      const uint8_t* xu = xp + u * xstep;
      static_for<2>([&](auto B) {
        constexpr int b = B.value;
        f32x4_t t[Q6 ? 2 : 1];
        static_for<4>([&](auto E) {
          constexpr int e = E.value, ti = Q6 ? e / 2 : 0;
          const f16x8_t c = mf_codes<SCH, b, e>(r);
          const bool first = Q6 ? e % 2 == 0 : e == 0;
#pragma unroll
          for (int n = 0; n < NH; n++) {
            const f16x8_t x = *reinterpret_cast<const f16x8_t*>(xu + ((B1 * b * 4 + e) * FS + n * MR) * 16);
            t[ti] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x, c, first && n == 0 ? zero : t[ti], 0, 0, 0);
          }
        });
        float s, m = 0.f;
        if constexpr (SCH == SCH_Q4_1) {
          s = f16_bits_to_f32(r.c[5 * b] & 0xffffu);
          m = f16_bits_to_f32(r.c[5 * b] >> 16);
        } else if constexpr (SCH == SCH_Q8_0) {
          s = f16_bits_to_f32(b ? r.c[8] >> 16 : r.c[0] & 0xffffu);
        } else if constexpr (MLX) {
          s = __uint_as_float(a.sb_bf16 ? r.h[b] << 16 : r.h[b]);
          m = __uint_as_float(a.sb_bf16 ? r.h[2 + b] << 16 : r.h[2 + b]);
        } else if constexpr (SCH == SCH_Q4_K) {
          // GGML's 6-bit packing: scales 0..3 and mins 0..3 in the low 6 bits
          // of bytes 0..7, scales and mins 4..7 in the nibbles of bytes 8..11
          // with their top two bits above the first ones'
          const uint32_t sc = g & 2 ? (r.h[3] & 0x0F0F0F0Fu) | ((r.h[1] >> 2) & 0x30303030u) : r.h[1] & 0x3F3F3F3Fu;
          const uint32_t mn = g & 2 ? ((r.h[3] >> 4) & 0x0F0F0F0Fu) | ((r.h[2] >> 2) & 0x30303030u) : r.h[2] & 0x3F3F3F3Fu;
          const uint32_t sh = 16 * (g & 1) + 8 * b;
          s = f16_bits_to_f32(r.h[0] & 0xffffu) * (float)((sc >> sh) & 0xffu);
          m = -f16_bits_to_f32(r.h[0] >> 16) * (float)((mn >> sh) & 0xffu);
        }
        // lane group g's block: 8u + 2g + b (Q6_K: as its codes)
        float inv[MR], sum[MR];
        mf_record<MR, HM>(recs, sums, 8 * u + (Q6 ? 4 * (g >> 1) + (g & 1) : 2 * g) + B1 * b, inv, sum);
        if constexpr (Q6) {
          const float d = f16_bits_to_f32(r.h[2]);
          const float s0 = d * (float)(int8_t)(r.h[b] & 0xffu), s1 = d * (float)(int8_t)(r.h[b] >> 8);
#pragma unroll
          for (int q = 0; q < MS; q++) acc[q] = fmaf(inv[q % MR], fmaf(s1, t[1][q], s0 * t[0][q]), acc[q]);
        } else {
#pragma unroll
          for (int q = 0; q < MS; q++) acc[q] = fmaf(s * inv[q % MR], t[0][q], acc[q]);
        }
        if constexpr (HM) {
#pragma unroll
          for (int q = 0; q < MR; q++) acc[q] = fmaf(m, sum[q], acc[q]);
        }
      });
      if (++cu == cnt) {
        // the tile's K is done: the lane groups' sums, then the waves', added
        // in wave order by one of them.  (Two buffers: the next tile's go to
        // the other one, and the one after's only behind the barrier that
        // follows this one's reads.)
        cu = 0;
#pragma unroll
        for (int q = 0; q < MS; q++) acc[q] = mf_rows(acc[q], [](float p, float q) { return p + q; });
        float v = acc[0];
#pragma unroll
        for (int q = 1; q < MS; q++) v = g == q ? acc[q] : v;
        red[(buf * W + wv) * 64 + lane] = v;   // lane 16 slot + j
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (turn == wv && g < MR) {
          float o = 0.f;
#pragma unroll
          for (int w = 0; w < W; w++) {
            o += red[(buf * W + w) * 64 + lane];
            if constexpr (MS > MR) o += red[(buf * W + w) * 64 + lane + 16 * MR];
          }
          const int64_t n = tile_row(ct) + j;
          if (g < a.M) {
            if (a.y_bf16) reinterpret_cast<uint16_t*>(a.y)[g * a.y_ld + n] = (uint16_t)f32_to_bf16_bits(o);
            else reinterpret_cast<float*>(a.y)[g * a.y_ld + n] = o;
          }
        }
        turn = (turn + 1) & (W - 1);
        buf ^= 1;
        ct += gridDim.x;
#pragma unroll
        for (int q = 0; q < MS; q++) acc[q] = 0.f;
      }
    });
  }
}

}  // namespace rlxq

#define RLXQ_MF_INST(NAME, SCH, XBF, MR, D)                                               \
  extern "C" __global__ __launch_bounds__(512, 4) void NAME(rlxq_gemv_args a) {          \
    rlxq::mf_body<SCH, XBF, MR, D>(a);                                                    \
  }
// (D units in flight per wave; six, with one workgroup per CU and twice the
// registers, were slower everywhere: Q8_0 12288->4096 13.0 us and 15.0)
#define RLXQ_MF_SCHEME(PRE, SCH, D)              \
  RLXQ_MF_INST(PRE##_mf_M1, SCH, true, 1, D)     \
  RLXQ_MF_INST(PRE##_mf_M2, SCH, true, 2, D)     \
  RLXQ_MF_INST(PRE##_mf_M4, SCH, true, 4, D)     \
  RLXQ_MF_INST(PRE##_mf1_F, SCH, false, 1, D)    \
  RLXQ_MF_INST(PRE##_mf2_F, SCH, false, 2, D)    \
  RLXQ_MF_INST(PRE##_mf4_F, SCH, false, 4, D)
RLXQ_MF_SCHEME(rlxq_gemvxs_q4_1, SCH_Q4_1, 3)
RLXQ_MF_SCHEME(rlxq_gemvxs_q4_k, SCH_Q4_K, 3)
RLXQ_MF_SCHEME(rlxq_gemvxs_mlx4, SCH_MLX4, 3)
RLXQ_MF_SCHEME(rlxq_gemv_q8_0, SCH_Q8_0, 2)
RLXQ_MF_SCHEME(rlxq_gemv_q6_k, SCH_Q6_K, 2)
