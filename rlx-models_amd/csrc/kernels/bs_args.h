/* Argument blocks of the block-scaled MFMA kernels (bsgemm.hip), shared by
 * the host (g++) and device (hipcc) compilers: plain C types only. */
#ifndef RLXQ_BS_ARGS_H
#define RLXQ_BS_ARGS_H
#include <stdint.h>

/* Activation preparation: f32 x [M, K] -> f16 MFMA fragments, each row scaled
 * by a power of two (inv_s[m] = 1 / scale) in two parts: the rounded row (hi)
 * and what the rounding left over (lo).
 * Fragment (block b of 32 elements, tile t of 32 rows, half m of the block,
 * part p) is 1 KB at (((b * rtiles + t) * 2 + m) * 2 + p) * 1024: lane
 * 32 h + j holds positions 16m + 8h .. + 7 (code order) of row 32 t + j.
 * Blocks run to kb8 (whole units of eight), rows to 32 rtiles; what lies
 * past K and M is zero.
 * ssum: the rows' block sums as f16 hi | lo << 16, for the min / bias term:
 * block 8 C + 4 h + q of row 32 t + j at dword
 * ((C * rtiles + t) * 64 + 32 h + j) * 4 + q.                              */
typedef struct rlxq_bs_prep_args {
  const float* x;
  uint8_t* x16;
  float* inv_s;           /* [32 rtiles]                                   */
  uint32_t* ssum;         /* [kb8 / 8][rtiles][64][4]                     */
  const int32_t* rmap;    /* row r is x row rmap[r] / rdiv, unused where
                             rmap[r] < 0; NULL: x row r                  */
  const int32_t* cmap;    /* with rmap: cmap[0] 32-row tiles are in use  */
  int64_t M, K;
  int32_t rtiles, kb8, order, rdiv;
} rlxq_bs_prep_args;

typedef struct rlxq_bs_args {
  const uint8_t* x16;     /* prepared fragments                            */
  const float* inv_s;
  const uint32_t* ssum;   /* block sums (formats with a min / bias)        */
  const uint8_t* w;       /* packed rows, row stride rb bytes              */
  const void* scales;     /* MLX: [N, K / group] (f32, or bf16), else NULL */
  const void* biases;
  float* part;            /* [splits, M, N] partial sums (splits > 1)      */
  void* y;                /* [M, N] output (splits == 1)                   */
  int64_t M, N, K, rb, y_ld, group;
  int32_t rtiles;         /* 32-row tiles of x16                           */
  int32_t uslice, splits; /* 256-element units per K split                 */
  int32_t tiles_n, tiles_m;
  int32_t y_bf16, sb_bf16, pad;
} rlxq_bs_args;

#endif
