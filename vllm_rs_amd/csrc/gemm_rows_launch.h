// gemm_rows_launch.h — the row-major prompt GEMM (gemm_rows.cuh) as the C entry points and the native runtime call it.
#pragma once
#include <type_traits>

#include "gemm_rows.cuh"

struct GemmRowsOut {
  void* out;
  const void* bias;
  int ld;
};
struct GemmRowsCall {
  const void* x = nullptr;
  int x_ld = 0, M = 0, K = 0;
  int nseg = 1;
  const void* w[GR_MAX_SEG] = {};  // dual: gate, up
  int n[GR_MAX_SEG] = {};
  const void* bias[GR_MAX_SEG] = {};
  void* out[GR_MAX_SEG] = {};  // dual: out[0] = silu(gate) * up
  int out_ld[GR_MAX_SEG] = {};
  const void* residual = nullptr;  // added to segment 0
  int res_ld = 0;
  int out_f32 = 0;
  bool dual = false;
  int tile = 0;  // rows / 64 * 16 + columns / 64 instead of gemm_rows_tile's choice
};
// whether the product can run here and is expected to be faster than on kernel B (and behind it the element-wise launches the fused form
// saves).  Measured, bf16, weights from memory, us (here / kernel B): 64 rows x 8192, K = 11008 89 / 66; 128 x 4096, K = 5632 41 / 38; 192 x 2048, K = 2048 17 / 20;
// 192 x 4096, K = 14336 98 / 112; 256 x 2048, K = 8192 52 / 42; 384 x 2048, K = 8192 51 / 64; beyond, the fused forms win: 2120 x 5632, K = 2048 95 / 219
bool vra_gemm_rows_fits(const GemmRowsCall& c);
bool vra_gemm_rows_takes(const GemmRowsCall& c);  // whether it can
void vra_launch_gemm_rows(const GemmRowsCall& c, int dtype, int64_t stream);
