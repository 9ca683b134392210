// Launches of the few-rows W4A16 MFMA kernel (w4_few_rows.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

struct FewRowsArgs {
  const uint16_t* x;         // bf16 activation rows of K
  const int64_t* perm;       // mode 1: x row of p = perm[p] / topk; mode 2: output row of p = perm[p]
  int topk;
  const uint32_t* w;         // int4pack [E, K, N/8]
  const uint16_t* s;         // bf16 scales [E, G, N]
  int K, N, gs;
  const int* tile_expert;    // row-tile table (nullptr: dense, one expert, R rows)
  const int* tile_row0;
  const int* tile_rows;
  const int* tile_count;
  int mtiles_max;            // row tiles the table has room for
  int R;
  uint16_t* y;
  int ldy;
  int MI;                    // mode 1: act width
  const uint16_t* wts;       // mode 2: bf16 routing weights, flat
};

constexpr int kFewRowsTile = 12;     // most rows of a table tile
constexpr int kFewRowsMaxK = 4096;   // fp16 rows of a tile stay in LDS

bool w4_few_rows_ok(int K, int N, int gs);
// mode 0: y bf16 [R, N] (tile table); 1: SwiGLU act; 2: weighted products
int launch_w4_few_rows(int mode, const FewRowsArgs& a, hipStream_t st);
// dense rows (no table)
int launch_w4_few_rows_dense(const FewRowsArgs& a, hipStream_t st);
