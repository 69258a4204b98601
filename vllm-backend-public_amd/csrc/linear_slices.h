// The form of linear_tiled on fp8 weights in which K is split over a workgroup's waves and x goes straight to registers (linear_slices.hip).
#pragma once
#include "common.h"

namespace mi355 {

struct LinearSlices {
  uint16_t* y;
  int64_t y_stride;
  float* partial;                  // [k groups][M][N]
  const uint16_t* x;
  int64_t x_stride;
  const void* w;                   // 1 KB blocks [K / 128][tiles][2]
  const float* w_scale;            // a row's, in tiled order
  const uint16_t* bias;
  int M, N, K, tiles, block_rows;  // block_rows: at most 32 but for M up to 32
};

// tp: tiles a workgroup; epilogue: 0 store, 1 SwiGLU, 2 partial sums.  False: there is no kernel for it.
bool launch_linear_slices(const LinearSlices& a, int tp, int k_groups, int epilogue, bool bf16, hipStream_t s);

}  // namespace mi355
