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
//   x Wq, x Wk, x Wv and y Wo    four (eight) lanes a column, a run of sixteen (eight) inner elements
//                                each, summed over the lanes by two (three) lane-crossing additions
//   q K^T                        the same lanes a cache row, 64 rows a pass
//   softmax and y = p V          every wave for its own columns: a lane takes one row of 64, so the
//                                exponentials of the rows are spread over the wave, and the sums over
//                                the rows halve the values as they double the lanes
// Only q, the new rows, the scores, y and x pass through LDS (64 values each, the scores one a row).
// Four waves, one a SIMD: what the loop spends is instructions (some 260 a step and wave, 4.4 clocks
// each, and 4 trips through LDS of 110), and the softmax is done in every wave; eight waves do it twice
// a SIMD.  Above 256 rows the caches fit the registers of eight waves only.
// 12 heads, 18 steps, us a launch, four waves : eight: 50 rows 22.0 : 24.3, 96 rows 26.3 : 28.8, 200 rows
// 35.0 : 37.6; 500 rows - : 57.0.  No step at 50 rows: 4.8, a step 0.93.
// The call at 50 rows: 2 450 us as host loop (some 180 launches), 22 as this kernel.  Error against 64
// bits over 17 sizes of 16 to 96 rows, mean: caches 1.8e-8, x 1.14e-7 (host loop 2.3e-8, 1.44e-7).
#include "../../../include/fxhip.h"
#include "fx_attn.h"
#include "fx_device.h"

namespace {
template <int CTRL>
__device__ __forceinline__ float dpp_get(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
template <int CTRL>
__device__ __forceinline__ int dpp_get(int v) { return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, false); }
// sum over the group of L = 4 or 8 neighbouring lanes, in all of them
template <int L>
__device__ __forceinline__ float lanes_sum(float v) {
  v += dpp_get<0xB1>(v);                            // quad_perm [1, 0, 3, 2]
  v += dpp_get<0x4E>(v);                            // quad_perm [2, 3, 0, 1]
  if constexpr (L == 8) v += dpp_get<0x141>(v);     // row_half_mirror: from lane 7 - l of the group of eight
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
// The largest value of the wave, in all lanes, by the order of the integers that floats are mapped to: a
// float maximum costs two more instructions a stage, which quiet operands from unknown sources.  (A NaN
// may win or lose: what is subtracted from or exponentiated is NaN either way.)
__device__ __forceinline__ float wave_max(float f) {
  int v = __float_as_int(f);
  v ^= (v >> 31) & 0x7fffffff;
  fx_u32x2s t = __builtin_amdgcn_permlane32_swap((unsigned)v, (unsigned)v, false, false);
  v = max((int)t.x, (int)t.y);
  t = __builtin_amdgcn_permlane16_swap((unsigned)v, (unsigned)v, false, false);
  v = max((int)t.x, (int)t.y);
  v = max(v, dpp_get<0x128>(v));   // row_ror:8
  v = max(v, dpp_get<0x141>(v));
  v = max(v, dpp_get<0xB1>(v));
  v = max(v, dpp_get<0x4E>(v));
  return __int_as_float(v ^ ((v >> 31) & 0x7fffffff));
}
__device__ __forceinline__ float wave_sum(float v) {
  float x, y;
  swap32(v, v, x, y);
  v = x + y;
  swap16(v, v, x, y);
  v = x + y;
  v += dpp_get<0x128>(v);
  return lanes_sum<8>(v);
}
// N = 8 or 16 values a lane in, one out: the sum over the wave of value lane / (64 / N).  Lanes that
// differ in one bit of their number add and keep half of the values each, from stage to stage.
template <int N>
__device__ __forceinline__ float wave_sums(const float (&p)[N], int lane) {
  float q[N / 2], r[N / 4], x, y;
#pragma unroll
  for (int i = 0; i < N / 2; ++i) {
    swap32(p[i], p[i + N / 2], x, y);
    q[i] = x + y;
  }
#pragma unroll
  for (int i = 0; i < N / 4; ++i) {
    swap16(q[i], q[i + N / 4], x, y);
    r[i] = x + y;
  }
  const bool b3 = (lane & 8) != 0;
  float s[N / 8];
#pragma unroll
  for (int i = 0; i < N / 8; ++i) {
    const float keep = b3 ? r[i + N / 8] : r[i], send = b3 ? r[i] : r[i + N / 8];
    s[i] = keep + dpp_get<0x128>(send);
  }
  if constexpr (N == 8) return lanes_sum<8>(s[0]);
  const bool b2 = (lane & 4) != 0;
  const float keep = b2 ? s[N / 8 - 1] : s[0], send = b2 ? s[0] : s[N / 8 - 1];
  return lanes_sum<4>(keep + dpp_get<0x141>(send));
}
template <int N>
__device__ __forceinline__ void load(float (&v)[N], const float* p) {
#pragma unroll
  for (int i = 0; i < N; i += 4) {
    const float4 f = *(const float4*)(p + i);
    v[i] = f.x; v[i + 1] = f.y; v[i + 2] = f.z; v[i + 3] = f.w;
  }
}
template <int N>
__device__ __forceinline__ void store(float* p, const float (&v)[N]) {
#pragma unroll
  for (int i = 0; i < N; i += 4) *(float4*)(p + i) = make_float4(v[i], v[i + 1], v[i + 2], v[i + 3]);
}
// (four sums side by side: a dependent product waits for the one before it)
template <int N>
__device__ __forceinline__ float dot(const float (&a)[N], const float (&b)[N]) {
  float s[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) s[i] = a[i] * b[i];
#pragma unroll
  for (int i = 4; i < N; ++i) s[i & 3] = __builtin_fmaf(a[i], b[i], s[i & 3]);
  return (s[0] + s[1]) + (s[2] + s[3]);
}
}  // namespace

// R: groups of 64 cache rows.  W: waves, and lanes that share a column or a cache row (N of its elements each).
template <int R, int W>
__global__ __launch_bounds__(W * 64) void fx_attention_kernel(const FxAttnArgs a) {
  constexpr int D = FX_ATTN_DEPTH, N = D / W;
  static_assert(W == 4 || W == 8, "sums over four or eight lanes");
  __shared__ __align__(16) float s_x[D], s_q[D], s_k[D], s_v[D], s_y[D], s_score[R * 64];
  const int lane = (int)threadIdx.x & 63, wave = (int)threadIdx.x >> 6;
  const int col = wave * N + lane / W;      // column of the products, and cache row of a group
  const int run = (lane % W) * N;           // first of the N inner elements of this lane
  const bool writes = lane % W == 0;
  const int head = (int)blockIdx.x % a.heads, rows = a.rows;
  const size_t w_at = (size_t)head * D * D + (size_t)run * D + col;
  float wq[N], wk[N], wv[N], wo[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    wq[i] = a.wq[w_at + (size_t)i * D];
    wk[i] = a.wk[w_at + (size_t)i * D];
    wv[i] = a.wv[w_at + (size_t)i * D];
    wo[i] = a.wo[w_at + (size_t)i * D];
  }
  // keys: row 64 j + col, N elements from run on; values: row 64 j + lane, columns N wave ... N wave + N - 1
  const size_t cache = (size_t)blockIdx.x * rows * D;
  float kc[R][N], vc[R][N];
#pragma unroll
  for (int j = 0; j < R; ++j) {
#pragma unroll
    for (int i = 0; i < N; ++i) kc[j][i] = vc[j][i] = 0.0f;
    if (64 * j + col < rows) {
      load(kc[j], a.k + cache + (size_t)(64 * j + col) * D + run);
#pragma unroll
      for (int i = 0; i < N; ++i) kc[j][i] += a.k_add;
    }
    if (64 * j + lane < rows) {
      load(vc[j], a.v + cache + (size_t)(64 * j + lane) * D + wave * N);
#pragma unroll
      for (int i = 0; i < N; ++i) vc[j][i] += a.v_add;
    }
  }
  if (threadIdx.x < D) s_x[threadIdx.x] = a.x[(size_t)blockIdx.x * D + threadIdx.x];
  __syncthreads();
  for (int s = 0; s < a.steps; ++s) {
    int row = a.start + s;   // a position below zero counts from the end (the caller has checked -rows <= row < rows)
    if (row < 0) row += rows;
    float in[N];
    load(in, s_x + run);
    const float q = lanes_sum<W>(dot(wq, in)), k = lanes_sum<W>(dot(wk, in)), v = lanes_sum<W>(dot(wv, in));
    if (writes) {
      s_q[col] = q;
      s_k[col] = k;
      s_v[col] = v;
    }
    __syncthreads();
    load(in, s_q + run);
#pragma unroll
    for (int j = 0; j < R; ++j) {
      if (64 * j + col == row) load(kc[j], s_k + run);
      if (64 * j + lane == row) load(vc[j], s_v + wave * N);
    }
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const float score = lanes_sum<W>(dot(kc[j], in)) * a.scale;
      if (writes) s_score[64 * j + col] = 64 * j + col < rows ? score : -__builtin_inff();
    }
    __syncthreads();
    // softmax(scores) V.  A row past the cache has score -inf, i.e. weight 0, and value 0.
    float e[R], sum = 0.0f, y[N];
#pragma unroll
    for (int j = 0; j < R; ++j) e[j] = s_score[64 * j + lane];
    float top = e[0];
#pragma unroll
    for (int j = 1; j < R; ++j) top = fmaxf(top, e[j]);
    top = wave_max(top);
#pragma unroll
    for (int j = 0; j < R; ++j) {
      e[j] = expf(e[j] - top) * (1.0f / (R * 64));   // (a power of two: the weights add up to no more than 1, so y is no larger than V)
      sum += e[j];
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
      y[i] = e[0] * vc[0][i];
#pragma unroll
      for (int j = 1; j < R; ++j) y[i] = __builtin_fmaf(e[j], vc[j][i], y[i]);
    }
    const float total = wave_sums(y, lane);
    if (writes) s_y[col] = total;
    const float per = 1.0f / wave_sum(sum);   // (applied behind Wo: the division runs while y travels)
    __syncthreads();
    load(in, s_y + run);
    const float next = lanes_sum<W>(dot(wo, in)) * per;
    if (writes) s_x[col] = next;
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < R; ++j) {
    if (64 * j + col < rows) store(a.k_out + cache + (size_t)(64 * j + col) * D + run, kc[j]);
    if (64 * j + lane < rows) store(a.v_out + cache + (size_t)(64 * j + lane) * D + wave * N, vc[j]);
  }
  if (threadIdx.x < D) a.x_out[(size_t)blockIdx.x * D + threadIdx.x] = s_x[threadIdx.x];
}

hipError_t fx_launch_attention_steps(const FxAttnArgs& a, int lanes, hipStream_t stream) {
  struct Form { const void* kernel; uint32_t threads; };
  const Form f = a.rows <= 64    ? Form{(const void*)fx_attention_kernel<1, 4>, 256}
                 : a.rows <= 128 ? Form{(const void*)fx_attention_kernel<2, 4>, 256}
                 : a.rows <= 256 ? Form{(const void*)fx_attention_kernel<4, 4>, 256}
                                 : Form{(const void*)fx_attention_kernel<8, 8>, 512};
  FxAttnArgs args = a;
  void* kargs[1] = {(void*)&args};
  return hipLaunchKernel(f.kernel, dim3((uint32_t)lanes), dim3(f.threads), kargs, 0, stream);
}
