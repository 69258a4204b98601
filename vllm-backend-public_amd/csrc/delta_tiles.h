// The gated delta rule over tiles of 16 rows (delta_tiles.hip) and chunks of 64 (delta_chunks.hip), called by mi355_gated_delta_rule.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mi355 {

struct DeltaTiles {
  float* o;                     // [rows][H][dv]
  const void *qkv, *beta, *decay;
  int64_t stride, beta_stride, decay_stride;
  const float *a_log, *dt_bias;
  float* state;                 // [slots][H][d][dv]
  const int32_t *cu_seqlens, *state_slots;
  const int64_t* positions;
  float* ws;
  int64_t rows;
  int q_off, k_off, v_off, per_channel, S, H, G, d, dv;
};

// floats of workspace: a decay per head needs about a third of what one per channel does
int64_t delta_tiles_workspace(int64_t rows, int H, int d, bool per_channel);
// dtype: an mi355_dtype code; d at most 256
void launch_delta_tiles(const DeltaTiles& a, int dtype, hipStream_t stream);

// floats of workspace of the form by chunks, 0 where it is not for these sizes; whether it takes these operands
int64_t delta_chunks_workspace(int64_t rows, int S, int H, int G, int d, bool per_channel);
bool delta_chunks_ok(const DeltaTiles& a, int dtype);
void launch_delta_chunks(const DeltaTiles& a, hipStream_t stream);

}  // namespace mi355
