// Single-query attention over a growing key / value cache as one launch (fx_attn.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define FX_ATTN_DEPTH 64      // elements of a head: its four 64 x 64 weights are 64 registers a lane of four waves
#define FX_ATTN_MAX_ROWS 512  // rows of a cache: both caches of a head are then 128 registers a lane of eight waves

// contiguous fp32 tensors, 16-byte aligned; see fx_attention_steps in include/fxhip.h
struct FxAttnArgs {
  const float *x, *k, *v;              // [lanes][64], [lanes][rows][64] twice; lane = batch row * heads + head
  const float *wq, *wk, *wv, *wo;      // [heads][64][64]
  float *k_out, *v_out, *x_out;
  int heads, rows, start, steps;
  float scale, k_add, v_add;
};
hipError_t fx_launch_attention_steps(const FxAttnArgs& a, int lanes, hipStream_t stream);
