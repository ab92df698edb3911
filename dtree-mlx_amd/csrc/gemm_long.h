// Interface between dtree_gemm_long's argument checks and its kernels.
#pragma once
#include "common.h"

namespace dtree {

struct LongParams {
  const uint16_t* x; const uint16_t* x_lo;
  const uint16_t* w; const uint16_t* w_sb; int rows, n, k;  // w_sb: q4 (scale, bias) pairs
  const float* ss_in; int ss_tiles; float inv_norm_dim; float eps;
  float* out_f32; int ld_out_f32;
  uint16_t* out_bf16; uint16_t* out_lo; int ld_out_bf16; int out_tiled;
  int out_h16;  // outputs in DTREE_W_TILED_F16: one fp16 plane
  const uint16_t* next_norm;
  float* ss_out;
  uint16_t* hidden_out; int ld_hidden;
  int ntn, tiles;  // column tiles, all tiles
  int vec;  // four consecutive elements of every operand may be moved as one vector
};

// Dense weights (bf16 with an optional low activation plane, or fp16); ntn and
// tiles are filled in here.
int launch_long_dense(LongParams p, int epi, bool h16, int cus, hipStream_t st);
int launch_long_q4(LongParams p, int epi, int cus, hipStream_t st);
// The tile the launches above choose, 1000 rows + columns.
int long_tile(bool q4, bool h16, bool lo, int epi, int rows, int n, int k, int cus);

}  // namespace dtree
