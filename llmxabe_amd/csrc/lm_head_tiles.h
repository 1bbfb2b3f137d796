// Interface of the LM head's launches for hidden sizes up to 2048 (lm_head_tiles.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace xabe {

struct LmHeadArgs {
  const uint8_t* w;
  const float* x;   // [*][K]
  float* out;       // [*][vocab]
  int K, vocab;
  int t0, nt;       // tokens [t0, t0 + nt) are served by this launch
  size_t w_bytes;   // quantized kernels: the tensor's length
  int seg_sb;       // k_lm_head_quant: superblocks whose activations LDS holds at a time
};

constexpr size_t kHeadTileTokens = 16;  // tokens per pass over the matrix
// Rows of two, four, six or eight superblocks: a wavefront of the workgroup for each.
inline bool head_tiles_width(size_t hidden) { return hidden % 512 == 0 && hidden <= 2048; }

int head_tiles_configure();
int launch_head_tiles_bf16(hipStream_t s, int num_cus, const LmHeadArgs& a);
int launch_head_tiles_q8(hipStream_t s, int num_cus, const LmHeadArgs& a);
int launch_head_tiles_q6k(hipStream_t s, int num_cus, const LmHeadArgs& a);

}  // namespace xabe
