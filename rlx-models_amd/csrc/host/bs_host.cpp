// Host side of the block-scaled MFMA matmul (f32 activations, from batched
// decode to prefill sizes): activation preparation, the matmul kernel, then
// (where K is split) the partial-sum reduction.
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "bs_args.h"
#include "rlxq.h"
#include "rlxq_internal.hpp"

namespace rlxq {

namespace {
size_t round256(size_t b) { return (b + 255) & ~(size_t)255; }
// Bytes of one weight row per 256-element unit.
int64_t bs_seg_bytes(int scheme) {
  switch (scheme) {
    case RLXQ_GGUF_Q4_1: return 160;
    case RLXQ_GGUF_Q4_0: case RLXQ_GGUF_Q4_K: return 144;
    case RLXQ_GGUF_Q8_0: return 272;
    case RLXQ_GGUF_Q5_K: return 176;
    case RLXQ_MLX_AFFINE4: return 128;
    case RLXQ_MLX_AFFINE8: return 256;
    case RLXQ_GGUF_Q6_K: return 240;   // (210 bytes from the dword they start in)
    default: return 0;
  }
}
// What a unit costs against Q4_1's (the codes' conversion and scales).
double bs_unit_factor(int scheme) {
  switch (scheme) {
    case RLXQ_MLX_AFFINE4: return 1.4;
    case RLXQ_GGUF_Q6_K: case RLXQ_MLX_AFFINE8: return 1.5;
    default: return 1.0;
  }
}
// Scratch of one pass over `rows` rows: fragments, row factors, block sums,
// K-split partial sums.
struct BsBytes {
  size_t x, s, sum, part;
  BsBytes(int64_t rows, int RT, int64_t n, int64_t nu, int64_t splits) {
    const int64_t t = (rows + 32 * RT - 1) / (32 * RT) * RT;   // 32-row tiles
    x = round256((size_t)(32 * nu * t) * 1024);   // (f16 hi and lo)
    s = round256((size_t)t * 128);
    sum = round256((size_t)(nu * t) * 1024);
    part = splits > 1 ? round256((size_t)(splits * rows * n) * 4) : 0;
  }
  size_t all() const { return x + s + sum + part; }
};
}  // namespace

bool bs_scheme(int scheme) {
  return bs_seg_bytes(scheme) > 0;
}

// (rows an odd number of 16-byte pieces apart)
int64_t bs_lds_row(int scheme) {
  const int64_t seg = bs_seg_bytes(scheme);
  return (seg / 16) % 2 ? seg : seg + 16;
}

namespace {
// LDS of the dense form: three activation slots (two 32-element blocks each),
// the waves' weight regions.
size_t bs_lds_bytes(int scheme, int RT) {
  return (size_t)(3 * RT * 2) * 4096 + (size_t)(128 * bs_lds_row(scheme));
}
}  // namespace

// Whether f32 rows take the block-scaled matmul or the kernels it stands
// beside: the batched-decode kernels (17 to 256 rows) and the exact GEMM
// (prefill), which both pad K to 128 and 64 where this one takes whole
// 256-element units, and start up faster.  T: its tiles (32 rows up to 32, 64
// past them, by 128 columns), two of which share a CU (Q8_0 and MLX 8 bit: one).
// us here / there, Q4_1 unless named; over 20800 batched and 6100 prefill
// shapes (K 64 to 16384, N 64 to 24576) the rule is 0.1 to 0.6% behind the
// faster of the two, this kernel alone 0.5 to 5%, prefill of Q8_0 and MLX 8 bit
// 4 and 12%.  RLXQ_BS=0 turns it off, any other value on (bs_dispatch).
bool bs_applies(int scheme, int64_t m, int64_t k, int64_t n, bool prefill) {
  if (!bs_scheme(scheme)) return false;
  // (the K-quants have no other kernel for f32 rows at prefill)
  if (prefill && !is_gguf(scheme) && !is_mlx(scheme)) return true;
  if (const char* e = std::getenv("RLXQ_BS")) return std::strcmp(e, "0") != 0;
  const int64_t rows = m <= 32 ? 32 : 64, T = (m + rows - 1) / rows * ((n + 127) / 128);
  const bool part = k % 256 != 0, mlx8 = scheme == RLXQ_MLX_AFFINE8, q8 = scheme == RLXQ_GGUF_Q8_0;
  if (prefill) {
    // long K and few columns: preparation alone (4096 rows of 12288->128: 266
    // and 165), which re-reads rows past 4096 elements
    if (k > 8192 && n <= 256 && m > 1024) return false;
    // the exact GEMM's tiles of 128 rows, filled
    const bool full = m <= 256 && m % 128 == 0;
    if (mlx8) {
      // one workgroup a CU: a second round costs what the first did (1024 rows
      // of 4096->24576: 990 and 812; 512 of 1024->4096, one round: 31 and 37), a first one from K = 2048 too
      if (T > 256) return false;
      if (part) return k > 64 && !full;
      return m <= 64 || k <= 1024 || T <= (k <= 2048 ? 128 : 32);
    }
    if (!part || k >= 512) return true;
    // K = 64 is a quarter of a unit, 128 half of one (1024 rows of 64->4096:
    // 17.3 and 15.7, Q8_0 22.5 and 15.9; 128 rows of 128->4096: 10.5 and 9.4)
    if (q8) return T <= 256 && k > 64 && !(full && k <= 128);
    if (k == 64) return T <= 256 && !full;
    return !full || (k > 128 && T <= 256);
  }
  const bool xr = q8 || scheme == RLXQ_GGUF_Q4_0 || scheme == RLXQ_GGUF_Q5_K;   // register-streamed beside it
  if (mlx8 && m > 32 && ((T > 256 && 10 * T < 6 * 256 * ((T + 255) / 256)) || (part && k < 1024)))
    return false;   // a second round nearly empty (160 rows of 1792->12288: 78 and 61)
  // one to four tiles of a long K (64 rows of 16384->64: 24.5 and 20.2)
  if (k >= 8192) return T > (xr ? 1 : 4) || (m <= 32 && (k < 12288 || T > 1));
  if (k >= 1024) return true;
  // short K: from so many tiles on that the other one's rounds grow (64 rows of
  // 384->4096 13.3 and 10.8, 512->4096 12.3 and 11.5, 256->4096 9.7 and 9.6;
  // 256 rows of 384->4096 14.5 and 14.6, 384->8192 15.6 and 23.2).  32 rows
  // fill a tile of their own (256->4096: 8.2 and 9.5).
  if (xr) {
    if (T > 64) return true;
    if (m <= 32) return !part && !(q8 && k == 768 && T > 16);
    return T > 32 || k == 256 || (k == 128 && scheme == RLXQ_GGUF_Q4_0) || (k == 768 && T <= 12);
  }
  if (m <= 32) return !part || T > 128;
  if (part) return T > 128;
  return T > 64 || (k == 768 && T <= 32);
}

int bs_order(int scheme) { return scheme == RLXQ_GGUF_Q5_K ? 1 : sk_order(scheme); }

// Eight rows per workgroup once those fill the chip (2048 gathered rows of
// 2048: 12.8 us, against 18 with a row per workgroup), two below (512 rows of
// 4096 took 12.9 us eight a workgroup, 9.6 one).
int bs_prep(rlxq_ctx* ctx, const rlxq_bs_prep_args& p, void* stream) {
  const int64_t rows = (int64_t)32 * p.rtiles;
  const int per = rows >= 2048 ? 8 : 2;
  const char* name = per == 8 ? "rlxq_bs_prep8" : "rlxq_bs_prep2";
  hipFunction_t fn;
  if (int rc = get_fn(ctx, name, &fn)) return rc;
  rlxq_bs_prep_args a = p;
  void* args[] = {&a};
  return launch(ctx, fn, dim3((unsigned)(rows / per)), dim3(1024), 0, stream, args, name);
}

namespace {
// One pass: preparation, matmul, reduction.
int bs_pass(rlxq_ctx* ctx, int scheme, const float* x, const void* w, int64_t rb, int64_t m, int64_t k,
            int64_t n, void* y, int y_dtype, void* stream, const SkinnySb& sb, int RT, int64_t splits, int64_t uslice,
            const char* name) {
  const int64_t nu = (k + 255) / 256, tiles_m = (m + 32 * RT - 1) / (32 * RT), tiles_n = (n + 127) / 128;
  const int64_t rtiles = tiles_m * RT;
  const BsBytes b(m, RT, n, nu, splits);
  void* ws = nullptr;
  int rc;
  if ((rc = workspace(ctx, b.all(), &ws, stream))) return rc;
  char* wsb = static_cast<char*>(ws);

  rlxq_bs_prep_args p;
  std::memset(&p, 0, sizeof p);
  p.x = x;
  p.x16 = reinterpret_cast<uint8_t*>(wsb);
  p.inv_s = reinterpret_cast<float*>(wsb + b.x);
  p.ssum = reinterpret_cast<uint32_t*>(wsb + b.x + b.s);
  p.M = m;
  p.K = k;
  p.rtiles = (int32_t)rtiles;
  p.kb8 = (int32_t)(8 * nu);
  p.order = bs_order(scheme);
  p.rdiv = 1;
  if ((rc = bs_prep(ctx, p, stream))) return rc;
  hipFunction_t fn;

  rlxq_bs_args a;
  std::memset(&a, 0, sizeof a);
  a.x16 = p.x16;
  a.inv_s = p.inv_s;
  a.ssum = p.ssum;
  a.w = static_cast<const uint8_t*>(w);
  a.scales = sb.scales;
  a.biases = sb.biases;
  a.part = splits > 1 ? reinterpret_cast<float*>(wsb + b.x + b.s + b.sum) : nullptr;
  a.y = y;
  a.M = m;
  a.N = n;
  a.K = k;
  a.rb = rb;
  a.y_ld = n;
  a.group = sb.group;
  a.rtiles = (int32_t)rtiles;
  a.uslice = (int32_t)uslice;
  a.splits = (int32_t)splits;
  a.tiles_n = (int32_t)tiles_n;
  a.tiles_m = (int32_t)tiles_m;
  a.y_bf16 = y_dtype == RLXQ_BF16;
  a.sb_bf16 = sb.sb_bf16;
  if ((rc = get_fn(ctx, name, &fn))) return rc;
  void* args[] = {&a};
  const size_t lds = bs_lds_bytes(scheme, RT);
  if ((rc = launch(ctx, fn, dim3((unsigned)(tiles_m * tiles_n * splits)), dim3(256), lds, stream, args, name)))
    return rc;
  if (splits > 1) {
    rlxq_skinny_args r;
    std::memset(&r, 0, sizeof r);
    r.part = a.part;
    r.y = y;
    r.M = m;
    r.N = n;
    r.y_ld = n;
    r.splits = (int32_t)splits;
    r.y_bf16 = a.y_bf16;
    rc = splits_reduce(ctx, r, stream);
    if (!rc) ctx->last_kernel = name;
  }
  return rc;
}
}  // namespace

int bs_dispatch(rlxq_ctx* ctx, int scheme, const float* x, const void* w, int64_t rb, int64_t m,
                int64_t k, int64_t n, void* y, int y_dtype, void* stream, const SkinnySb& sb, bool prefill,
                size_t counted) {
  const int64_t cus = ctx->cu_count > 0 ? ctx->cu_count : 256;
  const int64_t nu = (k + 255) / 256;   // 256-element units
  // 64-row tiles past 32 rows (197 rows of Q4_K, 4096->24576: 131 us in four
  // of them, 151 in seven 32-row ones; 64 rows of Q4_1: 51 and 55); 128
  // columns.  RLXQ_BS="RT,splits" (tuning) sets the 32-row tiles per
  // workgroup (1 or 2; 0: the form with 64-bit row offsets) and, unless 0,
  // the K splits.
  // (32 weight rows past 4 GB: the form with 64-bit row offsets)
  bool wide = rb >= ((int64_t)1 << 27);
  int RT = m > 32 ? 2 : 1;
  int64_t want = 0;
  if (const char* e = std::getenv("RLXQ_BS")) {
    int a1, a2;
    if (std::sscanf(e, "%d,%d", &a1, &a2) == 2 && a1 >= 0 && a1 <= 2) {
      want = a2;
      if (a1 == 0) wide = true;
      else RT = a1;
    }
  }
  if (wide) RT = 1;
  if (prefill)
    if (const char* e = std::getenv("RLXQ_GEMM_SPLITS")) want = std::max(1, std::atoi(e));
  const int64_t tiles_m = (m + 32 * RT - 1) / (32 * RT), tiles_n = (n + 127) / 128;
  int64_t splits = 1;
  if (want > 0) {
    splits = std::min<int64_t>(want, nu);
  } else {
    // K splits by what the rounds of workgroups cost: a 64-row unit takes
    // about 2.65 us per workgroup and CU (3.1 alone on the CU) times the
    // format's factor, a 32-row one 1.6 (1.9), the reduction 3.5 us and the
    // partial sums' traffic at about 5 TB/s.  At most 24 MiB of partial sums.
    // Over 180 shapes a format (K 512 to 12288, N 128 to 24576, 32 to 512 rows)
    // the choice is 0.3 to 0.8% behind the best of the measured splits.  (One
    // factor for all, and two workgroups a CU where the LDS holds one, Q8_0 and
    // MLX 8 bit: up to 2%, at worst 22%, 256 rows of Q6_K 4096->8192, 97 us and
    // 80.)
    const double f = RT == 2 ? bs_unit_factor(scheme) : 1.0;
    const bool two = 2 * bs_lds_bytes(scheme, RT) <= ctx->max_lds;
    double best = 1e30;
    for (int64_t t = 1; t <= 32 && t <= nu; t++) {
      const int64_t us = (nu + t - 1) / t, sp = (nu + us - 1) / us;
      if (sp != t || (t > 1 && t * m * n * 4 > ((int64_t)24 << 20))) continue;
      const int64_t per_cu = (tiles_m * tiles_n * t + cus - 1) / cus;
      const double unit = RT == 2 ? (two && per_cu > 1 ? 2.65 : 3.1) : (two && per_cu > 1 ? 1.6 : 1.9);
      const double cost = (double)(per_cu * us) * unit * f + (t > 1 ? 3.5 + (double)(t * m * n) * 8 / 5e6 : 0.0);
      if (cost < best) best = cost, splits = t;
    }
  }
  const int64_t uslice = (nu + splits - 1) / splits;
  splits = (nu + uslice - 1) / uslice;
  if (tiles_m * tiles_n * splits > 0x7fffffff || tiles_m * RT > 0x3ffffff)
    return fail(ctx, RLXQ_E_SHAPE, "dequant_matmul: block-scaled grid");

  // Rows per pass: all of them, or as many whole tiles as the array of the
  // no-allocation entry point holds (rows do not depend on each other and the
  // K splits stay those of the whole call: the same bits).  Which calls that
  // entry point takes is decided by `counted`, what the batched-decode kernels
  // or the exact GEMM need for them; fragments in whole 256-element units are
  // four times that at K = 64, and partial sums of other splits.
  int64_t pass = m;
  if (ctx->fixed_active) {
    if (counted > ctx->fixed_bytes) return scratch_refused(ctx, counted);
    if (BsBytes(m, RT, n, nu, splits).all() > ctx->fixed_bytes) {
      if (BsBytes(32 * RT, RT, n, nu, splits).all() > ctx->fixed_bytes) RT = 1;
      int64_t lo = 0, hi = (m + 32 * RT - 1) / (32 * RT);   // tiles that fit, and that do not
      while (hi - lo > 1) {
        const int64_t mid = (lo + hi) / 2;
        (BsBytes(mid * 32 * RT, RT, n, nu, splits).all() <= ctx->fixed_bytes ? lo : hi) = mid;
      }
      // (at prefill one does: 32 rows take half of what 64, the fewest, count)
      if (lo > 0) pass = lo * 32 * RT;
      else if (!prefill) return skinny_dispatch(ctx, scheme, x, RLXQ_F32, w, rb, m, k, n, y, y_dtype, stream, sb);
    }
  }
  char name[64];
  if (wide) std::snprintf(name, sizeof name, "rlxq_bs_%s_wide", scheme_name(scheme));
  else std::snprintf(name, sizeof name, "rlxq_bs_%s_rt%d", scheme_name(scheme), RT);
  int rc = RLXQ_OK;
  for (int64_t r0 = 0; r0 < m && !rc; r0 += pass)
    rc = bs_pass(ctx, scheme, x + r0 * k, w, rb, std::min(pass, m - r0), k, n, static_cast<char*>(y) + r0 * n * (y_dtype == RLXQ_BF16 ? 2 : 4), y_dtype,
                 stream, sb, RT, splits, uslice, name);
  return rc;
}

}  // namespace rlxq
