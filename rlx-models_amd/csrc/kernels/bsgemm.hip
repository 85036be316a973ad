// Block-scaled MFMA matmul for f32 activations over packed weights:
// y[m, n] = sum_k x[m, k] * dequant(W)[n, k], from 17 rows to prefill sizes, and
// the expert ops' gathered rows.
// Serves Op::DequantMatMul and Op::DequantGroupedMatMul on the reference's operand
// types (F32 x and y, crates/rlx-models-core/src/standard_decoder.rs:727-738,
// 12421-12433).
//
// A weight block is scale * code + min: the codes are integers that f16 holds
// exactly, so they go to the matrix cores as they are and the block's scale
// is applied in f32 to the block's 32 x 32 MFMA result:
//   T = sum over the block's two halves of mfma(x hi, codes) + mfma(x lo,
//   codes); acc += scale * T
// with one f32 scale per lane (lane j of a result holds column j).  Against
// carrying every weight as two f16 operands (hi and lo) that is two products
// per weight for f32 activations instead of three or four, and no conversion
// of weights beyond picking the code bits out.  (The code bits themselves as
// subnormal f16, code * 2^-24, would save the offset's addition, but the
// matrix cores align such products by their exponent field and lose about ten
// bits of the sum: 3e-6 against 2e-7 off float64.)  The min / bias term is
// one or two more MFMAs per 256 elements on the rows' prepared block sums.
// Q6_K has a scale per 16 weights, which is a block's half: code * scale as
// an f16 and what its rounding left (exact), three products.
//
// A wave owns 32 weight rows: their 256-element unit is read as row-contiguous
// 16-byte pieces one unit ahead and laid into the wave's own LDS region, from
// where lane (j, h) = (lane % 32, lane / 32) takes the code dwords of
// positions 8h .. and 16 + 8h .. of row j.  The activation fragments of a
// step (two blocks) are shared by the workgroup's four waves through LDS.
//
// What bounds it: the issue slots beside the MFMAs (per half-block MFMA about
// four VALU instructions: the scale FMAs and the unpacking) and LDS reads of
// the activation fragments; 30-35% of the MFMA rate.  Measured with f32 x and
// y, activation preparation and split-K sums included: Q4_1 4096->24576 at 64
// rows 90 -> 53 us, at 512 rows 377 -> 260 us; Q4_K at 197 rows 310 -> 131 us.
#include "common.hip.h"
#include "bs_args.h"
#include "f16dq.hip.h"
#include "gemm_dq.hip.h"
#include "moe_args.h"

namespace rlxq {

typedef float f32x16_t __attribute__((ext_vector_type(16)));

// Unit of the weight stream: 256 elements (8 blocks) of a row, PPR 16-byte
// pieces; rows LROW bytes apart in LDS (an odd number of 16-byte pieces, so
// that 16 rows' reads at one offset spread over the banks).
template <int SCH> constexpr int bs_seg() {
  return SCH == SCH_Q4_1 ? 160 : SCH == SCH_Q4_0 ? 144 : SCH == SCH_Q8_0 ? 272 : SCH == SCH_Q4_K ? 144
         : SCH == SCH_Q5_K ? 176 : SCH == SCH_MLX4 ? 128 : SCH == SCH_MLX8 ? 256 : SCH == SCH_Q6_K ? 208 : 0;
}
// (Q6_K: 210-byte super-blocks at 2-byte alignment, read from the dword they
// start in: 13 pieces and a last dword)
template <int SCH> constexpr int bs_lrow() {
  if (SCH == SCH_Q6_K) return 240;
  return (bs_seg<SCH>() / 16) % 2 ? bs_seg<SCH>() : bs_seg<SCH>() + 16;
}
template <int SCH> constexpr bool bs_mlx() { return SCH == SCH_MLX4 || SCH == SCH_MLX8; }
template <int SCH> constexpr bool bs_kq() { return SCH == SCH_Q4_K || SCH == SCH_Q5_K; }
// Operands per half-block: code, or for Q6_K code * scale as f16 hi and lo.
template <int SCH> constexpr int bs_nop() { return SCH == SCH_Q6_K ? 2 : 1; }
template <int SCH> constexpr bool bs_has_m() { return sk_has_m<SCH>(); }
// Power of two on the f16 min / bias halves (sk_wscale: MLX's f32 biases).
template <int SCH> constexpr float bs_mscale() { return 1.f / sk_wscale<SCH>(); }

// lo: what the lower 32 lanes held in v, hi: what the upper 32 held.
RLXQ_DEV void lane_halves(uint32_t v, uint32_t& lo, uint32_t& hi) {
  typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
  const u32x2_t p = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_permlane32_swap(v, v, false, false));
  lo = p.x;
  hi = p.y;
}

RLXQ_DEV uint32_t lds_u32(const uint8_t* p) { return *reinterpret_cast<const uint32_t*>(p); }

// What a lane keeps of one weight row over a unit: the K-quants' packed
// 6-bit scales and d, Q5_K's high bits, MLX's eight block scales; mn: the
// min / bias of blocks 4h .. 4h + 3 as f16 hi | lo << 16.
template <int SCH>
struct BsRow {
  uint32_t sa, sb, d;
  uint32_t qh[4];   // (Q6_K: the 16 int8 scales)
  uint32_t off;     // (Q6_K: 0 or 2, the super-block's first byte in the region)
  uint32_t sc[bs_mlx<SCH>() ? 8 : 1];
  uint32_t mn[4];
};
// A block as read from LDS: code dwords (raw) and the header dword.
template <int SCH>
struct BsRaw {
  uint32_t c[SCH == SCH_Q6_K ? 12 : 6], h;
};

// Reads the row's unit header (rp: the row in LDS; lane half h).
template <int SCH>
RLXQ_DEV void bs_row_head(const uint8_t* rp, int h, BsRow<SCH>& r) {
  if constexpr (SCH == SCH_Q6_K) {
    uint32_t w[5];
#pragma unroll
    for (int q = 0; q < 5; q++) w[q] = lds_u32(rp + 192 + 4 * q);
#pragma unroll
    for (int q = 0; q < 4; q++) r.qh[q] = align_bytes(w[q + 1], w[q], r.off);
    r.d = __float_as_uint(f16_bits_to_f32((w[4] >> (8 * r.off)) & 0xffffu));
  } else if constexpr (SCH == SCH_Q4_1) {
#pragma unroll
    for (int q = 0; q < 4; q++) r.mn[q] = lds_u32(rp + 80 * h + 20 * q) >> 16;
  } else if constexpr (bs_kq<SCH>()) {
    const u32x4_t hd = *reinterpret_cast<const u32x4_t*>(rp);
    // GGML's 6-bit packing: scales 0..3 and mins 0..3 in the low 6 bits of
    // bytes 0..7, scales and mins 4..7 in the nibbles of bytes 8..11 with
    // their top two bits above the first ones'
    r.sa = hd.y & 0x3F3F3F3Fu;
    r.sb = (hd.w & 0x0F0F0F0Fu) | ((hd.y >> 2) & 0x30303030u);
    const uint32_t ma = hd.z & 0x3F3F3F3Fu, mb = ((hd.w >> 4) & 0x0F0F0F0Fu) | ((hd.z >> 2) & 0x30303030u);
    r.d = __float_as_uint(f16_bits_to_f32(hd.x & 0xffffu));
    const float dm = -f16_bits_to_f32(hd.x >> 16);
    const uint32_t m4 = h ? mb : ma;
#pragma unroll
    for (int q = 0; q < 4; q++) r.mn[q] = f16_split(dm * (float)((m4 >> (8 * q)) & 0xffu));
    if constexpr (SCH == SCH_Q5_K) {
#pragma unroll
      for (int q = 0; q < 4; q++) r.qh[q] = lds_u32(rp + 16 + 4 * h + 8 * (q >> 1) + 16 * (q & 1));
    }
  }
}

// Block b (0..7, compile time) of the row as raw dwords: those holding the
// codes of positions 8h .. 8h + 7 and 16 + 8h .. 16 + 8h + 7.
template <int SCH, int b>
RLXQ_DEV void bs_fetch(const uint8_t* rp, int h, const BsRow<SCH>& r, BsRaw<SCH>& q) {
  if constexpr (SCH == SCH_Q4_1) {
    q.h = lds_u32(rp + 20 * b);
    q.c[0] = lds_u32(rp + 20 * b + 4 + 4 * h);
    q.c[1] = lds_u32(rp + 20 * b + 12 + 4 * h);
  } else if constexpr (SCH == SCH_Q4_0) {
    // even blocks start dword aligned (their codes 2 bytes further), odd
    // ones 2 bytes past it (codes aligned)
    if constexpr (b % 2 == 0) {
      q.h = lds_u32(rp + 18 * b);
#pragma unroll
      for (int i = 0; i < 4; i++) q.c[i] = lds_u32(rp + 18 * b + 4 * h + 8 * (i >> 1) + 4 * (i & 1));
    } else {
      q.h = lds_u32(rp + 18 * b - 2);
      q.c[0] = lds_u32(rp + 18 * b + 2 + 4 * h);
      q.c[1] = lds_u32(rp + 18 * b + 10 + 4 * h);
    }
  } else if constexpr (SCH == SCH_Q8_0) {
    if constexpr (b % 2 == 0) {
      q.h = lds_u32(rp + 34 * b);
#pragma unroll
      for (int i = 0; i < 6; i++) q.c[i] = lds_u32(rp + 34 * b + 8 * h + 16 * (i / 3) + 4 * (i % 3));
    } else {
      q.h = lds_u32(rp + 34 * b - 2);
#pragma unroll
      for (int i = 0; i < 4; i++) q.c[i] = lds_u32(rp + 34 * b + 2 + 8 * h + 16 * (i >> 1) + 4 * (i & 1));
    }
  } else if constexpr (bs_kq<SCH>()) {
    constexpr int o = (SCH == SCH_Q4_K ? 16 : 48) + 32 * (b / 2);
#pragma unroll
    for (int i = 0; i < 4; i++) q.c[i] = lds_u32(rp + o + 4 * h + 8 * (i >> 1) + 16 * (i & 1));
  } else if constexpr (SCH == SCH_Q6_K) {
    // ql bytes 64 (b / 4) + 32 (b % 2) .., qh bytes 32 (b / 4) .. (three
    // dwords per eight bytes: the region's bytes lie r.off further)
#pragma unroll
    for (int i = 0; i < 6; i++) {
      q.c[i] = lds_u32(rp + 64 * (b / 4) + 32 * (b & 1) + 8 * h + 16 * (i / 3) + 4 * (i % 3));
      q.c[6 + i] = lds_u32(rp + 128 + 32 * (b / 4) + 8 * h + 16 * (i / 3) + 4 * (i % 3));
    }
  } else if constexpr (SCH == SCH_MLX4) {
    q.c[0] = lds_u32(rp + 16 * b + 4 * h);
    q.c[1] = lds_u32(rp + 16 * b + 8 + 4 * h);
  } else {
    static_assert(SCH == SCH_MLX8, "format");
#pragma unroll
    for (int i = 0; i < 4; i++) q.c[i] = lds_u32(rp + 32 * b + 8 * h + 16 * (i >> 1) + 4 * (i & 1));
  }
}

// The lane's operand of half m of block b: the codes of positions 16m + 8h ..
// + 7, exact in f16 (1024 + code by bit pattern, then the offset off).
template <int SCH, int b, int m>
RLXQ_DEV void bs_operand(const BsRaw<SCH>& q, const BsRow<SCH>& r, f16x8_t (&o)[bs_nop<SCH>()]) {
  uint32_t u0, u1;
  if constexpr (SCH == SCH_Q4_1 || SCH == SCH_Q4_0 || SCH == SCH_MLX4) {
    const uint32_t c = (SCH == SCH_Q4_0 && b % 2 == 0) ? align_bytes(q.c[2 * m + 1], q.c[2 * m], 2) : q.c[m];
    u0 = c & 0x0F0F0F0Fu;
    u1 = (c >> 4) & 0x0F0F0F0Fu;
  } else if constexpr (bs_kq<SCH>()) {
    u0 = (q.c[2 * m] >> (4 * (b & 1))) & 0x0F0F0F0Fu;
    u1 = (q.c[2 * m + 1] >> (4 * (b & 1))) & 0x0F0F0F0Fu;
    if constexpr (SCH == SCH_Q5_K) {
      u0 |= (b < 4 ? r.qh[2 * m] << (4 - b) : r.qh[2 * m] >> (b - 4)) & 0x10101010u;
      u1 |= (b < 4 ? r.qh[2 * m + 1] << (4 - b) : r.qh[2 * m + 1] >> (b - 4)) & 0x10101010u;
    }
  } else if constexpr (SCH == SCH_Q8_0) {
    u0 = (b % 2 == 0 ? align_bytes(q.c[3 * m + 1], q.c[3 * m], 2) : q.c[2 * m]) ^ 0x80808080u;
    u1 = (b % 2 == 0 ? align_bytes(q.c[3 * m + 2], q.c[3 * m + 1], 2) : q.c[2 * m + 1]) ^ 0x80808080u;
  } else if constexpr (SCH == SCH_Q6_K) {
    // code (0..63) + 96 per byte, so that code - 32 = byte - 128
    constexpr int sl = 4 * ((b & 3) >> 1), sh = 2 * (b & 3);
    const uint32_t l0 = align_bytes(q.c[3 * m + 1], q.c[3 * m], r.off), l1 = align_bytes(q.c[3 * m + 2], q.c[3 * m + 1], r.off);
    const uint32_t h0 = align_bytes(q.c[3 * m + 7], q.c[3 * m + 6], r.off), h1 = align_bytes(q.c[3 * m + 8], q.c[3 * m + 7], r.off);
    u0 = (((l0 >> sl) & 0x0F0F0F0Fu) | (((h0 >> sh) & 0x03030303u) << 4)) + 0x60606060u;
    u1 = (((l1 >> sl) & 0x0F0F0F0Fu) | (((h1 >> sh) & 0x03030303u) << 4)) + 0x60606060u;
  } else {
    u0 = q.c[2 * m];
    u1 = q.c[2 * m + 1];
  }
  const _Float16 off = SCH == SCH_Q4_0 ? (_Float16)-1032.f
                       : (SCH == SCH_Q8_0 || SCH == SCH_Q6_K) ? (_Float16)-1152.f
                                                               : (_Float16)-1024.f;
  const f16x2_t o2 = {off, off};
  f16x2_t w[4] = {magic_lo(u0) + o2, magic_hi(u0) + o2, magic_lo(u1) + o2, magic_hi(u1) + o2};
  if constexpr (SCH == SCH_Q6_K) {
    // the half's int8 scale 2b + m: code * scale rounded to f16, and the rest
    // (an integer of at most 13 bits: both exact)
    const _Float16 sc = (_Float16)(float)(int8_t)((r.qh[b / 2] >> (8 * (2 * (b & 1) + m))) & 0xffu);
    const f16x2_t s2 = {sc, sc};
    f16x2_t v[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const f16x2_t p = w[i] * s2;
      v[i] = __builtin_elementwise_fma(w[i], s2, -p);
      w[i] = p;
    }
    o[bs_nop<SCH>() - 1] = f16x8_t{v[0].x, v[0].y, v[1].x, v[1].y, v[2].x, v[2].y, v[3].x, v[3].y};
  }
  o[0] = f16x8_t{w[0].x, w[0].y, w[1].x, w[1].y, w[2].x, w[2].y, w[3].x, w[3].y};
}

// The block's f32 scale.
template <int SCH, int b>
RLXQ_DEV float bs_scale(const BsRaw<SCH>& q, const BsRow<SCH>& r) {
  float s;
  if constexpr (SCH == SCH_Q4_1) s = f16_bits_to_f32(q.h & 0xffffu);
  else if constexpr (SCH == SCH_Q4_0 || SCH == SCH_Q8_0) s = f16_bits_to_f32(b % 2 ? q.h >> 16 : q.h & 0xffffu);
  else if constexpr (bs_kq<SCH>()) s = __uint_as_float(r.d) * (float)(((b < 4 ? r.sa : r.sb) >> (8 * (b & 3))) & 0xffu);
  else if constexpr (SCH == SCH_Q6_K) s = __uint_as_float(r.d);
  else s = __uint_as_float(r.sc[b]);
  // (kept in f32: folded into the FMAs as a mixed-precision operand it would
  // be converted again by each of them)
  asm volatile("" : "+v"(s));
  return s;
}

// The contraction of 32 RT activation rows (32-row tiles rt0 ..) with the
// wave's 32 TN weight rows (row r of them at w + roff(r)) over units [u0, u1).
// lds: three activation slots of 8 RT KB, then the four waves' weight
// regions of 32 TN LROW bytes.  Off: type of the byte offsets between the
// wave's weight rows (32 bits while 32 rows lie within 4 GB).
template <int SCH, int RT, int TN, class Off, class RowOff>
RLXQ_DEV void bs_core(const rlxq_gemm_args& ga, RowOff roff, const uint8_t* x16, const uint32_t* ssum, int rtiles,
                      int rt0, int u0, int u1, f32x16_t (&acc)[RT][TN], uint8_t* lds) {
  constexpr int NH = 2;                           // f16 hi and lo of an activation row
  constexpr int XB = RT * NH * 2;                 // fragments (1 KB) per block
  constexpr int SLOT = 2 * XB * 1024, NX = 2 * XB * 64 / 256;   // NX pieces per thread and step
  constexpr int SEG = bs_seg<SCH>(), PPR = SEG / 16, LROW = bs_lrow<SCH>(), R = 32 * TN;
  constexpr int NP = R * PPR, NL = (NP + 63) / 64;
  constexpr bool HM = bs_has_m<SCH>(), MLX = bs_mlx<SCH>();
  static_assert(SEG > 0 && SEG % 16 == 0 && NX >= 1, "unit");
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 31, h = lane >> 5;
  uint8_t* reg = lds + 3 * SLOT + wv * (R * LROW);

  // activation pieces of a step (two blocks): block i's XB fragments are
  // contiguous
  const u32x4_t* xg = reinterpret_cast<const u32x4_t*>(x16);
  const int64_t bstep = (int64_t)rtiles * NH * 128;   // pieces per block of x16
  int xoff[NX];   // (pieces; a step spans 2 bstep of them)
#pragma unroll
  for (int p = 0; p < NX; p++) {
    const int pc = tid + 256 * p;
    xoff[p] = (int)((pc / (64 * XB)) * bstep) + rt0 * NH * 128 + pc % (64 * XB);
  }
  const int s1 = 4 * u1 - 1;   // last step
  // steps of activations in flight to registers (two spilled for Q6_K and Q8_0)
  constexpr int XD = SCH == SCH_Q6_K || SCH == SCH_Q8_0 ? 1 : 2;
  u32x4_t xr[XD][NX];
  auto load_x = [&](int s, auto Q) {
    const u32x4_t* xs = xg + 2 * (int64_t)(s < s1 ? s : s1) * bstep;
#pragma unroll
    for (int p = 0; p < NX; p++) xr[Q.value][p] = xs[xoff[p]];
  };
  auto put_x = [&](int so, auto Q) {
#pragma unroll
    for (int p = 0; p < NX; p++) *reinterpret_cast<u32x4_t*>(lds + so + (tid + 256 * p) * 16) = xr[Q.value][p];
  };
  // weight pieces of a unit, in row order: piece p is 16-byte unit p % PPR of
  // row p / PPR
  // (byte offsets from the wave's first row)
  const uint8_t* wbase = ga.w + roff(0);
  Off src[NL];
  int dst[NL];
#pragma unroll
  for (int u = 0; u < NL; u++) {
    const int p = lane + 64 * u < NP ? lane + 64 * u : NP - 1;
    src[u] = (Off)(roff(p / PPR) - roff(0)) + (p % PPR) * 16;
    dst[u] = (p / PPR) * LROW + (p % PPR) * 16;
  }
  const Off tsrc = SCH == SCH_Q6_K ? (Off)(roff(j) - roff(0)) : 0u;
  u32x4_t wr[NL];
  uint32_t tail = 0u;   // Q6_K: the last dword of row j
  float ms[MLX ? TN : 1][4], mb[MLX ? TN : 1][4];
  const int ufull = (int)(ga.K / 256);   // units wholly inside K
  const int nblk = (int)(ga.K / 32);
  auto load_w = [&](int u) {
    const int uu = u < u1 ? u : u1 - 1;
    const uint8_t* ws = wbase + (int64_t)uu * SEG;
    if constexpr (SCH == SCH_Q6_K) {
      static_assert(TN == 1, "a row's last dword per lane");
      // (K is whole units.)  Row offsets are even: the dword a super-block
      // starts in lies 0 or 2 bytes before it, and everything read here stays
      // inside the super-block and those two bytes
      const Off uo = (Off)((reinterpret_cast<uintptr_t>(wbase) & 3u) + (uint64_t)uu * 210);
      const uint8_t* w4 = wbase - (reinterpret_cast<uintptr_t>(wbase) & 3u);
#pragma unroll
      for (int q = 0; q < NL; q++) {
        const uint32_t c = dst[q] % LROW;
        const uint4 v = ld_u128(w4 + ((src[q] - c + uo) & ~(Off)3) + c);
        wr[q] = u32x4_t{v.x, v.y, v.z, v.w};
      }
      const Off so = tsrc + uo, so4 = so & ~(Off)3;
      const uint16_t* p = reinterpret_cast<const uint16_t*>(w4 + so4 + 208);
      const uint32_t lo = p[0], hi = p[so & 2u ? 1 : 0];
      tail = lo | (hi << 16);
      return;
    }
    if (uu < ufull) {
#pragma unroll
      for (int q = 0; q < NL; q++) {
        const uint4 v = ld_u128(ws + src[q]);
        wr[q] = u32x4_t{v.x, v.y, v.z, v.w};
      }
    } else {
      // the last unit of a K that is not whole units: dwords past the row's
      // end read as zero (zero scales, zero weights)
#pragma unroll
      for (int q = 0; q < NL; q++) {
        const int p = lane + 64 * q < NP ? lane + 64 * q : NP - 1;
        const int64_t ro = (int64_t)uu * SEG + (p % PPR) * 16;
#pragma unroll
        for (int e = 0; e < 4; e++) wr[q][e] = ro + 4 * e + 4 <= ga.rb ? ld_u32(ws + src[q] + 4 * e) : 0u;
      }
    }
    if constexpr (MLX) {
      // scales and biases of blocks 4h .. 4h + 3 of the lane's rows
#pragma unroll
      for (int t = 0; t < TN; t++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const int kb = 8 * uu + 4 * h + q;
          const int64_t gi = roff.slab(32 * t + j) + ((int64_t)(kb < nblk ? kb : nblk - 1) * 32) / ga.group;
          float s, b;
          if (ga.sb_bf16) {
            s = bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(ga.scales)[gi]);
            b = bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(ga.biases)[gi]);
          } else {
            s = reinterpret_cast<const float*>(ga.scales)[gi];
            b = reinterpret_cast<const float*>(ga.biases)[gi];
          }
          ms[t][q] = kb < nblk ? s : 0.f;
          mb[t][q] = kb < nblk ? b : 0.f;
        }
    }
  };
  auto barrier = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

  const f32x16_t zero = {};
#pragma unroll
  for (int rt = 0; rt < RT; rt++)
#pragma unroll
    for (int t = 0; t < TN; t++) acc[rt][t] = zero;

  // Three activation slots: step s computes from one, step s + 1's lies
  // complete in the next (its first fragments are read during step s, so no
  // read waits behind a barrier), and step s + 2's, loaded a step earlier, is
  // stored into the third halfway through step s, so that the barrier at the
  // step's end finds the stores done.
  load_w(u0);
  static_for<2 / XD>([&](auto O) {   // steps 0 and 1, XD at a time
    static_for<XD>([&](auto I) { load_x(4 * u0 + O.value * XD + I.value, I); });
    static_for<XD>([&](auto I) { put_x((O.value * XD + I.value) * SLOT, I); });
  });
  // (step s's register set is (s - 2) % XD)
  static_for<XD>([&](auto I) { load_x(4 * u0 + 2 + I.value, I); });
  barrier();
  f16x8_t xa[2][RT][2][NH];   // fragments of a block and the next
  auto read_x = [&](auto BI, auto RI, int so) {
    const uint8_t* sl = lds + so + lane * 16;
#pragma unroll
    for (int m = 0; m < 2; m++)
#pragma unroll
      for (int e = 0; e < NH; e++)
        xa[BI.value][RI.value][m][e] =
            *reinterpret_cast<const f16x8_t*>(sl + (BI.value * XB + (RI.value * 2 + m) * NH + e) * 1024);
  };
  static_for<RT>([&](auto I) { read_x(std::integral_constant<int, 0>{}, I, 0); });
  int sc = 0, sn = SLOT, sp = 2 * SLOT;   // slots of steps s, s + 1, s + 2
  const uint8_t* rp[TN];
#pragma unroll
  for (int t = 0; t < TN; t++) rp[t] = reg + (32 * t + j) * LROW;

  for (int u = u0; u < u1; u++) {
    // the wave's region is its own: its stores and reads are ordered by the
    // wave's in-order LDS queue.  (Every lane stores, those past the last
    // piece that piece again: a conditional store would let the compiler move
    // the other lanes' reads before it.)
#pragma unroll
    for (int q = 0; q < NL; q++) *reinterpret_cast<u32x4_t*>(reg + dst[q]) = wr[q];
    BsRow<SCH> row[TN];
    if constexpr (SCH == SCH_Q6_K) {
      *reinterpret_cast<uint32_t*>(reg + j * LROW + 208) = tail;
      row[0].off = (uint32_t)((reinterpret_cast<uintptr_t>(wbase) & 3u) + (uint32_t)tsrc + (uint32_t)u * 210) & 2u;
    }
    if constexpr (MLX) {
#pragma unroll
      for (int t = 0; t < TN; t++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
          lane_halves(__float_as_uint(ms[t][q]), row[t].sc[q], row[t].sc[4 + q]);
          row[t].mn[q] = f16_split(mb[t][q] * sk_wscale<SCH>());
        }
    }
    asm volatile("" ::: "memory");
    load_w(u + 1);
    u32x4_t sf[HM ? RT : 1];
    if constexpr (HM) {
      const u32x4_t* sp = reinterpret_cast<const u32x4_t*>(ssum) + ((int64_t)u * rtiles + rt0) * 64 + lane;
#pragma unroll
      for (int rt = 0; rt < RT; rt++) sf[rt] = sp[rt * 64];
    }
#pragma unroll
    for (int t = 0; t < TN; t++) bs_row_head<SCH>(rp[t], h, row[t]);

    // The (block, column tile, row tile) triples in order, software-pipelined:
    // the scale FMAs of one triple's result, the next operand's unpacking and
    // the LDS reads further ahead sit between the MFMAs of this one.  (Left to
    // itself the compiler runs reads, MFMAs and FMAs one after the other.  The
    // 32 x 32 MFMA overlaps with VALU work of the other waves: 23 clocks for
    // one half of it with four FMAs against 30 for a 16 x 16 one with four,
    // two waves per SIMD.)
    BsRaw<SCH> raw[2];
    f16x8_t op[2][2][bs_nop<SCH>()];
    float fs[2];
    f32x16_t T[2];
    bs_fetch<SCH, 0>(rp[0], h, row[0], raw[0]);
    bs_fetch<SCH, 1 / TN>(rp[1 % TN], h, row[1 % TN], raw[1]);
    bs_operand<SCH, 0, 0>(raw[0], row[0], op[0][0]);
    bs_operand<SCH, 0, 1>(raw[0], row[0], op[0][1]);
    fs[0] = bs_scale<SCH, 0>(raw[0], row[0]);
    static_for<8 * TN * RT>([&](auto S) {
      constexpr int s = S.value, pr = s / RT, rt = s % RT, b = pr / TN, t = pr % TN, q = pr & 1, z = s & 1;
      // (the first pair of a block reads the next block's fragments)
      if constexpr (t == 0) {
        if constexpr (b % 2 == 0) read_x(std::integral_constant<int, 1>{}, std::integral_constant<int, rt>{}, sc);
        else read_x(std::integral_constant<int, 0>{}, std::integral_constant<int, rt>{}, sn);
      }
      if constexpr (rt == 0 && pr + 2 < 8 * TN) bs_fetch<SCH, (pr + 2) / TN>(rp[(pr + 2) % TN], h, row[(pr + 2) % TN], raw[q]);
      const f16x8_t(&xf)[2][NH] = xa[b & 1][rt];
      T[z] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xf[0][0], op[q][0][0], zero, 0, 0, 0);
      T[z] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xf[0][1], op[q][0][0], T[z], 0, 0, 0);
      T[z] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xf[1][0], op[q][1][0], T[z], 0, 0, 0);
      T[z] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xf[1][1], op[q][1][0], T[z], 0, 0, 0);
      if constexpr (bs_nop<SCH>() == 2) {   // (the lo x lo products, ~2^-22 of a term, are skipped)
        T[z] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xf[0][0], op[q][0][1], T[z], 0, 0, 0);
        T[z] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xf[1][0], op[q][1][1], T[z], 0, 0, 0);
      }
      if constexpr (s > 0) {
        constexpr int pp = (s - 1) / RT, rp1 = (s - 1) % RT, tp = pp % TN;
#pragma unroll
        for (int r = 0; r < 16; r++) acc[rp1][tp][r] = fmaf(T[z ^ 1][r], fs[pp & 1], acc[rp1][tp][r]);
      }
      if constexpr (pr + 1 < 8 * TN) {
        constexpr int nb = (pr + 1) / TN, nt = (pr + 1) % TN;
        if constexpr (RT == 1) {
          bs_operand<SCH, nb, 0>(raw[q ^ 1], row[nt], op[q ^ 1][0]);
          bs_operand<SCH, nb, 1>(raw[q ^ 1], row[nt], op[q ^ 1][1]);
          fs[q ^ 1] = bs_scale<SCH, nb>(raw[q ^ 1], row[nt]);
        } else {
          if constexpr (rt == RT - 2) bs_operand<SCH, nb, 0>(raw[q ^ 1], row[nt], op[q ^ 1][0]);
          if constexpr (rt == RT - 1) {
            bs_operand<SCH, nb, 1>(raw[q ^ 1], row[nt], op[q ^ 1][1]);
            fs[q ^ 1] = bs_scale<SCH, nb>(raw[q ^ 1], row[nt]);
          }
        }
      }
      static_for<2 * (NH + bs_nop<SCH>() - 1)>([&](auto V) {
        constexpr int rd = (t == 0 ? 1 : 0) + (rt == 0 ? 2 : 0);
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);                             // an MFMA
        if constexpr (rd > 0) __builtin_amdgcn_sched_group_barrier(0x100, rd, 0);    // LDS reads
        __builtin_amdgcn_sched_group_barrier(0x2, 8, 0);                             // VALU
      });
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (b % 2 == 0 && t == TN - 1 && rt == RT - 1) {
        constexpr std::integral_constant<int, (b / 2) % XD> Q{};
        put_x(sp, Q);
        load_x(4 * u + b / 2 + 2 + XD, Q);
      }
      if constexpr (b % 2 == 1 && t == TN - 1 && rt == RT - 1) {
        barrier();
        const int o = sc;
        sc = sn;
        sn = sp;
        sp = o;
      }
    });
    constexpr int sl = 8 * TN * RT - 1;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[RT - 1][TN - 1][r] = fmaf(T[sl & 1][r], fs[(sl / RT) & 1], acc[RT - 1][TN - 1][r]);
    if constexpr (HM) {
      // the unit's min / bias: lane half h's slots are blocks 4h .. 4h + 3,
      // each as (S hi, S lo) x (m hi, m hi), then x (m lo, m lo)
#pragma unroll
      for (int t = 0; t < TN; t++) {
        u32x4_t hi, lo;
#pragma unroll
        for (int q = 0; q < 4; q++) {
          hi[q] = perm_b32(row[t].mn[q], row[t].mn[q], 0x01000100u);
          lo[q] = perm_b32(row[t].mn[q], row[t].mn[q], 0x03020302u);
        }
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
          const f16x8_t sa = __builtin_bit_cast(f16x8_t, sf[rt]);
          if constexpr (bs_mscale<SCH>() == 1.f) {
            acc[rt][t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(sa, __builtin_bit_cast(f16x8_t, hi), acc[rt][t], 0, 0, 0);
            if constexpr (SCH != SCH_Q4_1)   // (Q4_1's m is an f16)
              acc[rt][t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(sa, __builtin_bit_cast(f16x8_t, lo), acc[rt][t], 0, 0, 0);
          } else {
            f32x16_t w = __builtin_amdgcn_mfma_f32_32x32x16_f16(sa, __builtin_bit_cast(f16x8_t, hi), zero, 0, 0, 0);
            w = __builtin_amdgcn_mfma_f32_32x32x16_f16(sa, __builtin_bit_cast(f16x8_t, lo), w, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 16; r++) acc[rt][t][r] = fmaf(w[r], bs_mscale<SCH>(), acc[rt][t][r]);
          }
        }
      }
    }
  }
}

// Byte offset (and MLX slab offset) of the wave's weight row r: rows past the
// last repeat it (their columns are not stored).
struct BsDenseRows {
  int64_t n0, N, rb, kg;
  RLXQ_DEV int64_t row(int r) const { return n0 + r < N ? n0 + r : N - 1; }
  RLXQ_DEV int64_t operator()(int r) const { return row(r) * rb; }
  RLXQ_DEV int64_t slab(int r) const { return row(r) * kg; }
};

// Dense form: workgroup = (32 RT rows, 128 TN weight rows, K split).
template <int SCH, int RT, int TN, class Off>
RLXQ_DEV void bs_body(const rlxq_bs_args& a) {
  extern __shared__ __align__(16) uint8_t bs_lds[];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j = lane & 31, h = lane >> 5;
  // Workgroup order: workgroups b, b + 8, ... run on one XCD (dealt round
  // robin); with a grid of whole eights each XCD takes a contiguous range of
  // the order below: bands of up to GM row tiles, inside a band row tiles
  // fastest, then column tiles, then splits, so that the weights the first
  // row tile reads from HBM the others find in that XCD's L2, with few
  // enough rows' activations between them to stay there too.
  constexpr int GM = 8;
  const int G = (int)gridDim.x;
  const int L = G % 8 == 0 ? (int)(blockIdx.x % 8) * (G / 8) + (int)(blockIdx.x / 8) : (int)blockIdx.x;
  const int band = GM * a.tiles_n * a.splits, first = L / band * GM, in = L % band;
  const int gm = a.tiles_m - first < GM ? a.tiles_m - first : GM;
  const int mc = first + in % gm, rest = in / gm;
  const int tn = rest % a.tiles_n, sp = rest / a.tiles_n;
  const int64_t n0 = (int64_t)tn * 128 * TN + wv * 32 * TN;
  const int nu = (int)((a.K + 255) / 256);
  const int u0 = sp * a.uslice, u1 = u0 + a.uslice < nu ? u0 + a.uslice : nu;
  rlxq_gemm_args ga;
  ga.w = a.w;
  ga.rb = a.rb;
  ga.K = a.K;
  ga.group = a.group;
  ga.sb_bf16 = a.sb_bf16;
  ga.scales = a.scales;
  ga.biases = a.biases;
  const BsDenseRows roff{n0, a.N, a.rb, bs_mlx<SCH>() ? a.K / a.group : 0};
  f32x16_t acc[RT][TN];
  bs_core<SCH, RT, TN, Off>(ga, roff, a.x16, a.ssum, a.rtiles, mc * RT, u0, u1, acc, bs_lds);
  // C[i][j] of a 32 x 32 tile sits in lane j + 32 ((i / 4) % 2), register
  // 4 (i / 8) + i % 4.  The row factors come as vector loads and the bounds
  // and the destination are decided once per workgroup (a load and a branch
  // per row cost 3 us, 16 dependent round trips).
  const int64_t mw = (int64_t)mc * 32 * RT, m0 = mw + 4 * h, nl = n0 + j;
  f32x4_t is[RT][4];
#pragma unroll
  for (int rt = 0; rt < RT; rt++)
#pragma unroll
    for (int q = 0; q < 4; q++) is[rt][q] = *reinterpret_cast<const f32x4_t*>(a.inv_s + m0 + 32 * rt + 8 * q);
  auto epi = [&](auto put, auto checked) {
    static_for<RT>([&](auto I) {
      static_for<TN>([&](auto J) {
#pragma unroll
        for (int r = 0; r < 16; r++) {
          const int dm = 32 * I.value + 8 * (r / 4) + r % 4;
          if (!checked.value || (m0 + dm < a.M && nl + 32 * J.value < a.N))
            put(dm, 32 * J.value, acc[I.value][J.value][r] * is[I.value][r / 4][r % 4]);
        }
      });
    });
  };
  const bool whole = mw + 32 * RT <= a.M && n0 + 32 * TN <= a.N;
  auto epi_any = [&](auto put) {
    if (whole) epi(put, std::false_type{});
    else epi(put, std::true_type{});
  };
  if (a.splits > 1) {
    float* p = a.part + ((int64_t)sp * a.M + m0) * a.N + nl;
    epi_any([&](int dm, int dn, float v) { p[(int64_t)dm * a.N + dn] = v; });
  } else if (a.y_bf16) {
    uint16_t* p = reinterpret_cast<uint16_t*>(a.y) + m0 * a.y_ld + nl;
    epi_any([&](int dm, int dn, float v) { p[(int64_t)dm * a.y_ld + dn] = (uint16_t)f32_to_bf16_bits(v); });
  } else {
    float* p = reinterpret_cast<float*>(a.y) + m0 * a.y_ld + nl;
    epi_any([&](int dm, int dn, float v) { p[(int64_t)dm * a.y_ld + dn] = v; });
  }
}

// Grouped (MoE) form for prefill-sized calls: a workgroup takes one chunk of 32
// gathered rows, all of one expert, and 128 weight rows of that expert's slab
// (SwiGLU: 128 gate rows and the matching up rows N / 2 further on, a wave's
// second column tile, and the epilogue writes silu(g) * u).  Output rows go to
// the rows' entries.  Replaces the backend kernel of Op::DequantGroupedMatMul
// and the MoE expert FFN (crates/rlx-models-core/src/standard_decoder.rs:
// 12634-12760) at prefill sizes with F32 activations.  Against 16-row MFMA
// tiles on hi / lo row pairs (8 entries per weight pass, four products) it is
// one weight pass per 32 entries and two products: a 256-token layer of Q4_K
// experts (2048 -> 1536 and 768 -> 2048, 16 entries per expert), gate|up 242
// -> 91 us, down 150 -> 57 us.
struct BsMoeRows {
  int64_t n0, width, rb, kg, e0;   // e0: the expert's first row of the bank
  RLXQ_DEV int64_t row(int r) const {
    const int64_t c = n0 + (r & 31) < width ? n0 + (r & 31) : width - 1;
    return r < 32 ? c : width + c;
  }
  RLXQ_DEV int64_t operator()(int r) const { return row(r) * rb; }
  RLXQ_DEV int64_t slab(int r) const { return (e0 + row(r)) * kg; }
};

template <int SCH, bool SW>
RLXQ_DEV void bs_moe_body(const rlxq_moe_sk_args& a) {
  constexpr int TN = SW ? 2 : 1;
  extern __shared__ __align__(16) uint8_t bs_lds[];
  // The grid is sized for the most chunks there can be: the chunks there are
  // go to the XCDs in contiguous ranges (workgroups b, b + 8, ... share one),
  // so that a chunk's activations stay in one L2.
  const int total = a.cmap[0] * a.tiles_n, per = (total + 7) / 8;
  const int L = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
  if ((int)(blockIdx.x / 8) >= per || L >= total) return;
  const int chunk = L / a.tiles_n, tn = L % a.tiles_n;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j = lane & 31, h = lane >> 5;
  const int e = a.cmap[1 + chunk];
  const int64_t width = SW ? a.N / 2 : a.N;
  const int64_t n0 = (int64_t)tn * 128 + wv * 32;
  rlxq_gemm_args ga;
  ga.w = a.bank + (int64_t)e * a.N * a.rb;
  ga.rb = a.rb;
  ga.K = a.K;
  ga.group = a.group;
  ga.sb_bf16 = a.sb_bf16;
  ga.scales = a.scales;
  ga.biases = a.biases;
  const BsMoeRows roff{n0, width, a.rb, bs_mlx<SCH>() ? a.K / a.group : 0, (int64_t)e * a.N};
  f32x16_t acc[1][TN];
  bs_core<SCH, 1, TN, uint32_t>(ga, roff, reinterpret_cast<const uint8_t*>(a.x16), reinterpret_cast<const uint32_t*>(a.ssum),
                         (int)(a.Mp / 32), chunk, 0, (int)((a.K + 255) / 256), acc, bs_lds);
  typedef int32_t i32x4_t __attribute__((ext_vector_type(4)));
  const int64_t m0 = (int64_t)chunk * 32 + 4 * h, c = n0 + j;
  i32x4_t ent[4];
  f32x4_t is[4];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    ent[q] = *reinterpret_cast<const i32x4_t*>(a.emap + m0 + 8 * q);
    is[q] = *reinterpret_cast<const f32x4_t*>(a.inv_s + m0 + 8 * q);
  }
  if (c >= width) return;
#pragma unroll
  for (int r = 0; r < 16; r++) {
    if (ent[r / 4][r % 4] < 0) continue;
    float o = acc[0][0][r] * is[r / 4][r % 4];
    if constexpr (SW) o = o / (1.f + expf(-o)) * (acc[0][TN - 1][r] * is[r / 4][r % 4]);
    const int64_t off = (int64_t)ent[r / 4][r % 4] * a.y_ld + c;
    if (a.y_bf16) reinterpret_cast<uint16_t*>(a.y)[off] = (uint16_t)f32_to_bf16_bits(o);
    else reinterpret_cast<float*>(a.y)[off] = o;
  }
}

// Activation preparation: a workgroup of 1024 threads for ROWS rows, 1024 /
// ROWS threads a row: thread t of a row on pieces t, t + PT, ... (piece = 8
// positions of a block), the first NP of them kept in registers between the
// row maximum and the conversion.  Eight rows fill whole 128-byte lines of
// the fragments (a line holds one piece of eight rows), which the L2 then
// writes back once; with a row per workgroup the lines' parts came from
// several XCDs: 2048 gathered rows of 2048 took 18 us.  Two rows a workgroup
// where rows are few and the work has to spread over the CUs.
template <int ORD, int ROWS>
RLXQ_DEV void bs_prep_body(const rlxq_bs_prep_args& a) {
  constexpr int PT = 1024 / ROWS, NP = ROWS == 8 ? 4 : 3, NW = PT / 64;
  __shared__ float red[16];
  const int t = threadIdx.x % PT, rw = __builtin_amdgcn_readfirstlane(threadIdx.x / PT), lane = threadIdx.x & 63;
  const int r = blockIdx.x * ROWS + rw;
  const int i = t & 3;   // the thread's piece of its blocks (PT is a multiple of 4)
  const int nblk = (int)(a.K / 32), np = a.kb8 * 4;
  int64_t src = r;
  bool live = r < a.M;
  if (a.rmap) {
    // (a gathered padding row's fragments are left as they are: they reach only
    // its own output row, which is not stored)
    if ((int)(blockIdx.x * ROWS) >= a.cmap[0] * 32) return;
    const int32_t ent = a.rmap[r];
    live = ent >= 0;
    src = (live ? ent : 0) / a.rdiv;
  }
  auto load = [&](int p, float* v) {
    const int b = p >> 2;
    if (b >= nblk) {
#pragma unroll
      for (int e = 0; e < 8; e++) v[e] = 0.f;
      return;
    }
    // positions 8i .. 8i + 7 in code order: natural, GGUF nibbles (elements
    // 4i .. 4i + 3, 16 + 4i ..), MLX nibbles (8i, 8i + 2, .., 8i + 1, ..)
    const int64_t e0 = src * a.K + (int64_t)b * 32 + (ORD == 1 ? 4 * i : 8 * i);
    const int64_t e1 = e0 + (ORD == 1 ? 16 : 4);
    const float4 f0 = *reinterpret_cast<const float4*>(a.x + e0), f1 = *reinterpret_cast<const float4*>(a.x + e1);
    const float n[8] = {f0.x, f0.y, f0.z, f0.w, f1.x, f1.y, f1.z, f1.w};
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = n[ORD == 2 ? (e < 4 ? 2 * e : 2 * (e - 4) + 1) : e];
  };
  float v[NP][8], amax = 0.f, s = 1.f, inv = 0.f;
  if (live) {
#pragma unroll
    for (int q = 0; q < NP; q++)
      if (t + PT * q < np) {
        load(t + PT * q, v[q]);
#pragma unroll
        for (int e = 0; e < 8; e++) amax = fmaxf(amax, fabsf(v[q][e]));
      }
    for (int p = t + PT * NP; p < np; p += PT) {
      float u[8];
      load(p, u);
#pragma unroll
      for (int e = 0; e < 8; e++) amax = fmaxf(amax, fabsf(u[e]));
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off, 64));
    if (lane == 0) red[threadIdx.x >> 6] = amax;
  }
  __syncthreads();
  if (live) {
#pragma unroll
    for (int w = 0; w < NW; w++) amax = fmaxf(amax, red[rw * NW + w]);
    // the power of two that puts the row maximum in [2^9, 2^10): a block sum
    // then stays below 2^15, inside f16
    inv = 1.f;
    if (amax > 0.f && amax <= 3.4e38f) {
      int sh = 9 - ilogbf(amax);
      sh = sh < -126 ? -126 : (sh > 126 ? 126 : sh);
      s = ldexpf(1.f, sh);
      inv = ldexpf(1.f, -sh);
    }
  }
  if (a.rmap && !live) return;
  if (t == 0) a.inv_s[r] = inv;
  const int rt = r >> 5, j = r & 31;
  auto put = [&](int p, const float* u) {
    const int b = p >> 2;
    uint32_t hi[4], lo[4];
    float sum = 0.f;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const float w0 = live ? u[2 * e] * s : 0.f, w1 = live ? u[2 * e + 1] * s : 0.f;
      const uint32_t h0 = f32_to_f16_bits(w0), h1 = f32_to_f16_bits(w1);
      hi[e] = h0 | (h1 << 16);
      // the remainder w - hi is exact in f32; rounded once more
      const float r0 = w0 - f16_bits_to_f32(h0), r1 = w1 - f16_bits_to_f32(h1);
      const uint32_t l0 = f32_to_f16_bits(r0), l1 = f32_to_f16_bits(r1);
      lo[e] = l0 | (l1 << 16);
      sum += w0;
      sum += w1;
    }
    // piece i: half i / 2 of the block, lane 32 (i % 2) + j
    uint4* dst = reinterpret_cast<uint4*>(a.x16) + ((((int64_t)b * a.rtiles + rt) * 2 + (i >> 1)) * 2) * 64 + 32 * (i & 1) + j;
    dst[0] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
    dst[64] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
    // the block's four pieces are four neighbouring lanes
    sum += __shfl_xor(sum, 1, 64);
    sum += __shfl_xor(sum, 2, 64);
    if (i == 0) a.ssum[(((int64_t)(b >> 3) * a.rtiles + rt) * 64 + 32 * ((b >> 2) & 1) + j) * 4 + (b & 3)] = f16_split(sum);
  };
#pragma unroll
  for (int q = 0; q < NP; q++)
    if (t + PT * q < np) put(t + PT * q, v[q]);
  for (int p = t + PT * NP; p < np; p += PT) {
    float u[8];
    if (live) load(p, u);
    put(p, u);
  }
}

}  // namespace rlxq

#if RLXQ_PART_IS(0)
#define RLXQ_BS_PREP(NAME, ROWS)                                                               \
  extern "C" __global__ __launch_bounds__(1024) void NAME(rlxq_bs_prep_args a) {               \
    if (a.order == 1) rlxq::bs_prep_body<1, ROWS>(a);                                          \
    else if (a.order == 2) rlxq::bs_prep_body<2, ROWS>(a);                                     \
    else rlxq::bs_prep_body<0, ROWS>(a);                                                       \
  }
RLXQ_BS_PREP(rlxq_bs_prep2, 2)
RLXQ_BS_PREP(rlxq_bs_prep8, 8)
#endif

// rlxq_bs_<scheme>_rt<RT>: 32 RT rows a workgroup.  rlxq_bs_<scheme>_wide:
// rows of 128 MB and more, whose offsets take 64 bits (a register more per
// piece: the others stay on 32).  rlxq_moesk_<scheme>_bs[_sw]: the grouped
// form, with SwiGLU.
#define RLXQ_BS_INST(NAME, SCH, RT, OFF)                                                       \
  extern "C" __global__ __launch_bounds__(256, 2) void NAME(rlxq_bs_args a) {                  \
    rlxq::bs_body<SCH, RT, 1, OFF>(a);                                                      \
  }
#define RLXQ_BS_SCHEME(SNAME, SCH)                                                             \
  RLXQ_BS_INST(rlxq_bs_##SNAME##_rt1, SCH, 1, uint32_t)                                         \
  RLXQ_BS_INST(rlxq_bs_##SNAME##_rt2, SCH, 2, uint32_t)                                         \
  RLXQ_BS_INST(rlxq_bs_##SNAME##_wide, SCH, 1, uint64_t)                                        \
  extern "C" __global__ __launch_bounds__(256, 2) void rlxq_moesk_##SNAME##_bs(rlxq_moe_sk_args a) { \
    rlxq::bs_moe_body<SCH, false>(a);                                                          \
  }
#define RLXQ_BS_SW(SNAME, SCH)                                                                 \
  extern "C" __global__ __launch_bounds__(256, 2) void rlxq_moesk_##SNAME##_bs_sw(rlxq_moe_sk_args a) { \
    rlxq::bs_moe_body<SCH, true>(a);                                                           \
  }
#if RLXQ_PART_IS(0)
RLXQ_BS_SCHEME(q4_1, SCH_Q4_1)
RLXQ_BS_SW(q4_1, SCH_Q4_1)
RLXQ_BS_SCHEME(mlx4, SCH_MLX4)
RLXQ_BS_SCHEME(mlx8, SCH_MLX8)
#endif
#if RLXQ_PART_IS(1)
RLXQ_BS_SCHEME(q4_0, SCH_Q4_0)
RLXQ_BS_SW(q4_0, SCH_Q4_0)
RLXQ_BS_SW(q8_0, SCH_Q8_0)
RLXQ_BS_SCHEME(q8_0, SCH_Q8_0)
#endif
#if RLXQ_PART_IS(2)
RLXQ_BS_SCHEME(q4_k, SCH_Q4_K)
RLXQ_BS_SW(q4_k, SCH_Q4_K)
RLXQ_BS_SW(q5_k, SCH_Q5_K)
RLXQ_BS_SCHEME(q5_k, SCH_Q5_K)
RLXQ_BS_SCHEME(q6_k, SCH_Q6_K)
#endif
