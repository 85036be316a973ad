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

int bs_dispatch(rlxq_ctx* ctx, int scheme, const void* x, int x_dtype, const void* w, int64_t rb, int64_t m,
                int64_t k, int64_t n, void* y, int y_dtype, void* stream, const SkinnySb& sb, bool prefill) {
  const int64_t cus = ctx->cu_count > 0 ? ctx->cu_count : 256;
  const int64_t nu = (k + 255) / 256;   // 256-element units
  // 64-row tiles past 32 rows (197 rows of Q4_K, 4096->24576: 131 us in four
  // of them, 151 in seven 32-row ones; 64 rows of Q4_1: 51 and 55); 128
  // columns.  RLXQ_BS="RT,splits" (tuning) sets the 32-row tiles per
  // workgroup (1 or 2; 0: the form with 64-bit row offsets) and, unless 0,
  // the K splits.
  const int64_t r32 = (m + 31) / 32;
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
  const int64_t rtiles = tiles_m * RT;
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
  if (tiles_m * tiles_n * splits > 0x7fffffff || rtiles > 0x3ffffff)
    return fail(ctx, RLXQ_E_SHAPE, "dequant_matmul: block-scaled grid");

  const int nh = 2;
  const size_t x_bytes = round256((size_t)(16 * nu * rtiles * nh) * 1024), s_bytes = round256((size_t)rtiles * 128);
  const size_t sum_bytes = round256((size_t)(nu * rtiles) * 1024);
  const size_t part_bytes = splits > 1 ? round256((size_t)(splits * m * n) * 4) : 0;
  void* ws = nullptr;
  int rc;
  // (what counts against the no-allocation limit: the f16 hi and lo rows)
  const size_t need = x_bytes + s_bytes + sum_bytes + part_bytes, core = (size_t)(r32 * 32 * k) * 4;
  if ((rc = workspace(ctx, need, &ws, stream, need > core ? need - core : 0))) return rc;
  char* wsb = static_cast<char*>(ws);

  rlxq_bs_prep_args p;
  std::memset(&p, 0, sizeof p);
  p.x = x;
  p.x16 = reinterpret_cast<uint8_t*>(wsb);
  p.inv_s = reinterpret_cast<float*>(wsb + x_bytes);
  p.ssum = reinterpret_cast<uint32_t*>(wsb + x_bytes + s_bytes);
  p.M = m;
  p.K = k;
  p.rtiles = (int32_t)rtiles;
  p.nh = nh;
  p.kb8 = (int32_t)(8 * nu);
  p.order = bs_order(scheme);
  p.x_bf16 = x_dtype == RLXQ_BF16;
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
  a.part = splits > 1 ? reinterpret_cast<float*>(wsb + x_bytes + s_bytes + sum_bytes) : nullptr;
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
  char name[64];
  if (wide) std::snprintf(name, sizeof name, "rlxq_bs_%s_wide", scheme_name(scheme));
  else std::snprintf(name, sizeof name, "rlxq_bs_%s_rt%d", scheme_name(scheme), RT);
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

}  // namespace rlxq
