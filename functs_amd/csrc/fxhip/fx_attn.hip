// A decoding loop of single-query attention over a growing cache
//   for s in [0, steps): q = x Wq; k[row] = x Wk; v[row] = x Wv (row = start + s)
//                        x = softmax(scale * q K^T) V Wo
// (functs/benchmark/simpleops/attention/attention.py:38-58) as ONE launch.  The reference runs the
// loop on the host: six library products and their glue a step.
//
// Bound: the chain of dependent steps; a step's arithmetic is some 20 k products a head.  Heads of
// different batch rows never meet, so a workgroup takes one head of one row through all steps and
// nothing crosses workgroups.  The four 64 x 64 weight matrices and both caches stay in registers
// for the whole loop (read once, the caches written once); a step is four products with a barrier
// behind each:
//   x Wq, x Wk, x Wv and x' Wo   eight lanes a column, a run of eight inner elements each, summed
//                                over the eight lanes by three data-parallel-primitive additions
//   q K^T                        eight lanes a cache row (64 rows a pass), the same way
//   softmax and p V              every wave for its own eight columns: a lane takes one row of 64, so
//                                the exponentials of the rows are spread over the wave, and the sums
//                                over the rows halve the values as they double the lanes
// Only q, the new key, the scores, x' and x pass through LDS (64 values each, the scores one a row).
// 12 heads, 50 rows, 18 steps: 2 412 us a call as host loop (some 180 launches), 26.3 us as this
// kernel, which fills all of that: 1.3 us a step.  Error against 64 bits over 17 sizes of 16 to 96 rows,
// mean: caches 1.8e-8, x 1.16e-7 (host loop 2.3e-8, 1.44e-7).
#include "../../../include/fxhip.h"
#include "fx_attn.h"
#include "fx_device.h"

namespace {
template <int CTRL>
__device__ __forceinline__ float dpp_get(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
// sum over the group of eight lanes, in all of them
__device__ __forceinline__ float sum8(float v) {
  v += dpp_get<0xB1>(v);    // quad_perm [1, 0, 3, 2]
  v += dpp_get<0x4E>(v);    // quad_perm [2, 3, 0, 1]
  v += dpp_get<0x141>(v);   // row_half_mirror: from lane 7 - l of the group of eight
  return v;
}
typedef unsigned fx_u32x2s __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void swap32(float a, float b, float& x, float& y) {
  const fx_u32x2s t = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  x = __uint_as_float(t.x);
  y = __uint_as_float(t.y);
}
__device__ __forceinline__ void swap16(float a, float b, float& x, float& y) {
  const fx_u32x2s t = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  x = __uint_as_float(t.x);
  y = __uint_as_float(t.y);
}
__device__ __forceinline__ float wave_max(float v) {
  float x, y;
  swap32(v, v, x, y);
  v = fmaxf(x, y);
  swap16(v, v, x, y);
  v = fmaxf(x, y);
  v = fmaxf(v, dpp_get<0x128>(v));   // row_ror:8
  v = fmaxf(v, dpp_get<0x141>(v));
  v = fmaxf(v, dpp_get<0xB1>(v));
  return fmaxf(v, dpp_get<0x4E>(v));
}
__device__ __forceinline__ float wave_sum(float v) {
  float x, y;
  swap32(v, v, x, y);
  v = x + y;
  swap16(v, v, x, y);
  v = x + y;
  v += dpp_get<0x128>(v);
  return sum8(v);
}
// Eight values a lane in: the sum over the wave of value lane >> 3 out.  Lanes that differ in one
// bit of lane >> 3 add and keep half of the values each.
__device__ __forceinline__ float wave_sum8(const float (&p)[8], int lane) {
  float q[4], r[2], x, y;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    swap32(p[i], p[i + 4], x, y);
    q[i] = x + y;
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    swap16(q[i], q[i + 2], x, y);
    r[i] = x + y;
  }
  const bool b3 = (lane & 8) != 0;
  const float keep = b3 ? r[1] : r[0], send = b3 ? r[0] : r[1];
  return sum8(keep + dpp_get<0x128>(send));
}
struct Eight { float v[8]; };
__device__ __forceinline__ Eight load8(const float* p) {
  const float4 a = *(const float4*)p, b = *(const float4*)(p + 4);
  return Eight{{a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w}};
}
__device__ __forceinline__ void store8(float* p, const float (&v)[8]) {
  *(float4*)p = make_float4(v[0], v[1], v[2], v[3]);
  *(float4*)(p + 4) = make_float4(v[4], v[5], v[6], v[7]);
}
__device__ __forceinline__ float dot8(const float (&a)[8], const Eight& b) {
  float s = a[0] * b.v[0];
#pragma unroll
  for (int i = 1; i < 8; ++i) s = __builtin_fmaf(a[i], b.v[i], s);
  return s;
}
}  // namespace

// R: groups of 64 cache rows
template <int R>
__global__ __launch_bounds__(512) void fx_attention_kernel(const FxAttnArgs a) {
  constexpr int D = FX_ATTN_DEPTH;
  __shared__ __align__(16) float s_x[D], s_q[D], s_k[D], s_y[D], s_score[R * 64];
  const int lane = (int)threadIdx.x & 63, wave = (int)threadIdx.x >> 6;
  const int col = wave * 8 + (lane >> 3);   // column of the products, and cache row of a group
  const int run = (lane & 7) * 8;           // first of the eight inner elements of this lane
  const int head = (int)blockIdx.x % a.heads, rows = a.rows;
  const size_t w_at = (size_t)head * D * D + (size_t)run * D + col;
  float wq[8], wk[8], wv[8], wo[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    wq[i] = a.wq[w_at + (size_t)i * D];
    wk[i] = a.wk[w_at + (size_t)i * D];
    wv[i] = a.wv[w_at + (size_t)i * D];
    wo[i] = a.wo[w_at + (size_t)i * D];
  }
  // keys: row 64 j + col, elements run ... run + 7; values: row 64 j + lane, columns 8 wave ... 8 wave + 7
  const size_t cache = (size_t)blockIdx.x * rows * D;
  const float *k_in = a.k + cache, *v_in = a.v + cache;
  float kc[R][8], vc[R][8];
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const bool k_live = 64 * j + col < rows, v_live = 64 * j + lane < rows;
    Eight kk{}, vv{};
    if (k_live) kk = load8(k_in + (size_t)(64 * j + col) * D + run);
    if (v_live) vv = load8(v_in + (size_t)(64 * j + lane) * D + wave * 8);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      kc[j][i] = k_live ? kk.v[i] + a.k_add : 0.0f;
      vc[j][i] = v_live ? vv.v[i] + a.v_add : 0.0f;
    }
  }
  if (threadIdx.x < D) s_x[threadIdx.x] = a.x[(size_t)blockIdx.x * D + threadIdx.x];
  __syncthreads();
  for (int s = 0; s < a.steps; ++s) {
    int row = a.start + s;   // a position below zero counts from the end (the caller has checked -rows <= row < rows)
    if (row < 0) row += rows;
    const Eight x = load8(s_x + run);
    const float q = sum8(dot8(wq, x)), kn = sum8(dot8(wk, x)), vn = sum8(dot8(wv, x));
    if ((lane & 7) == 0) {
      s_q[col] = q;
      s_k[col] = kn;
    }
    // the new value row: column col is known to the eight lanes of its group, lane row & 63 wants the wave's eight
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float c = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(vn), 8 * i));
#pragma unroll
      for (int j = 0; j < R; ++j) vc[j][i] = 64 * j + lane == row ? c : vc[j][i];
    }
    __syncthreads();
    const Eight qv = load8(s_q + run), kv = load8(s_k + run);
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const bool mine = 64 * j + col == row;
#pragma unroll
      for (int i = 0; i < 8; ++i) kc[j][i] = mine ? kv.v[i] : kc[j][i];
      const float score = sum8(dot8(kc[j], qv)) * a.scale;
      if ((lane & 7) == 0) s_score[64 * j + col] = 64 * j + col < rows ? score : -__builtin_inff();
    }
    __syncthreads();
    // softmax(scores) V.  A row past the cache has score -inf, i.e. weight 0, and value 0.
    float e[R], top = -__builtin_inff(), sum = 0.0f, y[8];
#pragma unroll
    for (int j = 0; j < R; ++j) {
      e[j] = s_score[64 * j + lane];
      top = fmaxf(top, e[j]);
    }
    top = wave_max(top);
#pragma unroll
    for (int j = 0; j < R; ++j) {
      e[j] = expf(e[j] - top);
      sum += e[j];
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      y[i] = e[0] * vc[0][i];
#pragma unroll
      for (int j = 1; j < R; ++j) y[i] = __builtin_fmaf(e[j], vc[j][i], y[i]);
    }
    sum = wave_sum(sum);
    const float total = wave_sum8(y, lane);
    if ((lane & 7) == 0) s_y[col] = total / sum;
    __syncthreads();
    const float next = sum8(dot8(wo, load8(s_y + run)));
    if ((lane & 7) == 0) s_x[col] = next;
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < R; ++j) {
    if (64 * j + col < rows) store8(a.k_out + cache + (size_t)(64 * j + col) * D + run, kc[j]);
    if (64 * j + lane < rows) store8(a.v_out + cache + (size_t)(64 * j + lane) * D + wave * 8, vc[j]);
  }
  if (threadIdx.x < D) a.x_out[(size_t)blockIdx.x * D + threadIdx.x] = s_x[threadIdx.x];
}

hipError_t fx_launch_attention_steps(const FxAttnArgs& a, int lanes, hipStream_t stream) {
  auto kernel = a.rows <= 64 ? fx_attention_kernel<1> : a.rows <= 128 ? fx_attention_kernel<2> : a.rows <= 256 ? fx_attention_kernel<4> : fx_attention_kernel<8>;
  FxAttnArgs args = a;
  void* kargs[1] = {(void*)&args};
  return hipLaunchKernel((const void*)kernel, dim3((uint32_t)lanes), dim3(512), kargs, 0, stream);
}
