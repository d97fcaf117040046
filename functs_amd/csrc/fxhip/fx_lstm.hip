// Persistent stacked-LSTM kernel: the whole (time, layer) loop nest of
//   for t: cur = x[t]; for j: gates = cur @ Wih[j] + bih[j] + h[j] @ Whh[j] + bhh[j];
//          c[j] = f * c[j] + i * g; h[j] = o * tanh(c[j]); cur = h[j];  out[t] = cur
// (functs/benchmark/ai_model/lstm/lstm.py:79-133) as ONE launch.  The reference runs this loop on
// the host, one fused kernel and two library GEMMs per (t, j).
//
// A workgroup owns FX_LSTM_UPW hidden units, i.e. 4 * FX_LSTM_UPW gate columns of every layer's
// two weight matrices.  The inner dimension is split over its threads: thread k holds row k of
// those columns, for every layer, IN REGISTERS for the whole sequence (the 16.8 MB of weights of
// the benchmark configuration are read from memory once), and in every step it fetches element k
// of the step's vectors itself: x[t][k] and, per layer, element k of the h written in the step
// before.  Nothing is staged: the products stay in the thread, 16 partial sums a thread (two
// layers) are summed over the wave by a butterfly that halves the number of values as it doubles
// the lanes summed (lane-swap and data-parallel-primitive instructions, no LDS), the waves' sums
// meet in LDS behind the step's one barrier, and sixteen lanes of the first wave add the biases,
// apply the gates and update the cells; the cell state never leaves its lane.
// Steps are the diagonals t + j of the loop nest.  There is no barrier between workgroups: an h
// value travels with the tag of the step that wrote it and readers poll for the tag they expect
// (fx_lstm_sched.h), with bounded waits.
#include <hip/hip_runtime.h>

#include <map>
#include <mutex>
#include <set>
#include <thread>
#include <utility>

#define FX_LSTM_HD __host__ __device__
#include "../../../include/fxhip.h"
#include "fx_device.h"
#include "fx_lstm_groups.h"
#include "fx_lstm_sched.h"

#define FX_LSTM_BLOCK 256
#define FX_LSTM_MAXB 16
#define FX_LSTM_UPW 2   // hidden units per workgroup
#ifndef FX_LSTM_FIRST_LOOK
#define FX_LSTM_FIRST_LOOK 8   // units of 64 clocks; 7 to 10 are within 4 % of each other on the benchmark shape, 0 and 16 cost 40 and 8 %
#endif
// hooks for timing the phases of a step in a test build; nothing in the library
#ifndef FX_LSTM_STAMP
#define FX_LSTM_STAMP(k)
#define FX_LSTM_PSTAMP(k)
#define FX_LSTM_POLLS(n)
#define FX_LSTM_STAMP_END()
#define FX_LSTM_STAMP_DECL
#endif

namespace {
// Everything that crosses workgroups (the tagged h values, the control words) is written and read
// with device-scope atomic accesses, which go through to the memory side of the caches: no
// release / acquire fences, which on this device would write back and invalidate whole caches
// once per step.  A tagged value is one 64-bit store, so a reader never sees a value without
// its tag.
struct DevAtomics {
  static __device__ __forceinline__ uint32_t add(uint32_t* p) {
    return __hip_atomic_fetch_add(p, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  static __device__ __forceinline__ uint32_t load(uint32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  static __device__ __forceinline__ void store(uint32_t* p, uint32_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  static __device__ __forceinline__ void store64(uint64_t* p, uint64_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
};

template <int CTRL>
__device__ __forceinline__ float dpp_get(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
// the value of lane K of the caller's group of four lanes
template <int K>
__device__ __forceinline__ float quad_lane(float v) { return dpp_get<K * 0x55>(v); }

typedef unsigned fx_u32x2v __attribute__((ext_vector_type(2)));
// Sixteen values a lane in, one out: lane l gets the sum over the wave of value l >> 2.  Every
// stage adds a value across two lanes that differ in one bit of the lane number and keeps only
// half of the values in each of them, so the work halves from stage to stage:
//   lanes l and l ^ 32 (the upper half keeps values 8-15), rows of 16 lanes r and r ^ 1 (odd rows
//   keep the upper half of what is left), lanes l and l ^ 8, lanes l and the mirrored lane of
//   their group of eight, and at last the four lanes of a group, which hold the same value.
__device__ __forceinline__ float wave_sum16(const float (&p)[16], int lane) {
  float q[8], r[4], s2[2];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const fx_u32x2v t = __builtin_amdgcn_permlane32_swap(__float_as_uint(p[i]), __float_as_uint(p[i + 8]), false, false);
    q[i] = __uint_as_float(t.x) + __uint_as_float(t.y);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const fx_u32x2v t = __builtin_amdgcn_permlane16_swap(__float_as_uint(q[i]), __float_as_uint(q[i + 4]), false, false);
    r[i] = __uint_as_float(t.x) + __uint_as_float(t.y);
  }
  const bool b3 = (lane & 8) != 0, b2 = (lane & 4) != 0;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const float keep = b3 ? r[i + 2] : r[i], send = b3 ? r[i] : r[i + 2];
    s2[i] = keep + dpp_get<0x128>(send);   // row_ror:8: from lane l ^ 8
  }
  const float keep = b2 ? s2[1] : s2[0], send = b2 ? s2[0] : s2[1];
  float v = keep + dpp_get<0x141>(send);   // row_half_mirror: from lane 7 - l of the group of eight
  v = v + dpp_get<0xB1>(v);                // quad_perm [1, 0, 3, 2]
  v = v + dpp_get<0x4E>(v);                // quad_perm [2, 3, 0, 1]
  return v;
}
}  // namespace

// 1024 hidden units (two elements a thread) are resident together only at four waves per SIMD,
// i.e. within 128 registers a lane; the smaller sizes need two
template <int L, int HPT, int UPW>
__global__ __launch_bounds__(FX_LSTM_BLOCK * UPW, HPT >= 32 ? 4 : 2) void fx_lstm_stack_kernel(const FxLstmArgs a) {
  static_assert(UPW == 2, "the butterfly sums 16 values: two layers of four gates of two units");
  constexpr int NT = FX_LSTM_BLOCK * UPW;                             // threads
  constexpr int NW = NT / 64;                                         // waves
  constexpr int HH = HPT * 32;                                        // H
  constexpr int EPT = (HH + NT - 1) / NT;                             // rows of the weights per thread
  constexpr int NG = (L + 1) / 2;                                     // pairs of layers: 16 values each
  __shared__ float s_part[2][NG][NW][16];   // the waves' sums, by parity of the (step, batch row) pair: read behind the
                                            // pair's barrier, written again two barriers later
  __shared__ float s_c[FX_LSTM_MAXB][64];   // cell states: [batch row][owner lane]
  __shared__ uint32_t s_abort;
  FX_LSTM_STAMP_DECL
  const int H = a.H, B = a.B, T = a.T;
  const int tid = (int)threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  FX_LSTM_PSTAMP(0);
  // Workgroups go to the chip's eight dies in turn, and every die has a cache of its own: the
  // workgroups of a die take neighbouring hidden units, so that a die fetches its eighth of every
  // weight row once (lines of a row are shared by 32 units) instead of every die fetching all of it.
  const int n_wg = (int)gridDim.x;
  const int wg = (n_wg % 8 == 0) ? ((int)blockIdx.x % 8) * (n_wg / 8) + (int)blockIdx.x / 8 : (int)blockIdx.x;
  const int u0 = wg * UPW;
  // a workspace that still carries a given-up wait is refused (below, behind the first barrier)
  if (tid == 0) s_abort = fx_lstm_refused<DevAtomics>(a) ? 1u : 0u;
  // tags of this launch start behind those of every launch before it
  const uint32_t base = DevAtomics::load(a.ctl + FX_LSTM_W_BASE);

  // rows k = tid + e * NT of the workgroup's columns: [layer][gate][unit], input and recurrent matrix
  float w_ih[L][4][UPW][EPT], w_hh[L][4][UPW][EPT];
#pragma unroll
  for (int j = 0; j < L; ++j)
#pragma unroll
    for (int g = 0; g < 4; ++g)
#pragma unroll
      for (int e = 0; e < EPT; ++e) {
        const int k = tid + e * NT;
        float2 wi = make_float2(0.0f, 0.0f), wh = wi;
        if (k < HH) {
          const size_t at = ((size_t)(j * 4 + g) * H + k) * H + u0;   // u0 is even: 8-byte aligned
          wi = *(const float2*)(a.wih + at);
          wh = *(const float2*)(a.whh + at);
        }
        w_ih[j][g][0][e] = wi.x; w_ih[j][g][1][e] = wi.y;
        w_hh[j][g][0][e] = wh.x; w_hh[j][g][1][e] = wh.y;
      }
  // Lane 4 * v + gate of the first wave ends up with the gate sum of value v = (layer in its pair,
  // unit) of every pair of layers; the lane of gate 0 owns the cell.
  const int f_v = lane >> 2, f_gate = lane & 3, f_ul = f_v & 1, f_jl = f_v >> 1;
  float f_bias_ih[NG], f_bias_hh[NG];
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    const int j = 2 * g + f_jl;
    const bool live = wave == 0 && lane < 16 && j < L;
    f_bias_ih[g] = live ? a.bih[(size_t)(j * 4 + f_gate) * H + u0 + f_ul] : 0.0f;
    f_bias_hh[g] = live ? a.bhh[(size_t)(j * 4 + f_gate) * H + u0 + f_ul] : 0.0f;
  }
  if (wave == 0) {
    for (int b = 0; b < B; ++b) {
      float c = 0.0f;
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        // one lane owns at most one cell per pair of layers; with two pairs the second pair's cells
        // live in lanes 16-31
        const int j = 2 * g + ((lane & 15) >> 3), ul = ((lane & 15) >> 2) & 1;
        if ((lane >> 4) == g && (lane & 3) == 0 && j < L && a.c0) c = a.c0[((size_t)j * B + b) * H + u0 + ul];
      }
      s_c[b][lane] = c;
    }
  }
  __syncthreads();
  if (s_abort != 0u) {   // uniform: written once, ahead of the barrier
    if (tid == 0 && a.err_host) __hip_atomic_store(a.err_host, (uint32_t)FX_ASYNC_BARRIER, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    fx_lstm_poison(a, L, (uint32_t)tid, (uint32_t)NT);
    return;
  }
  FX_LSTM_PSTAMP(1);

  const int n_steps = fx_lstm_steps(T, L);
  // x of the next (step, batch row) is asked for at the top of a step, ahead of the polls, and is
  // in its register long before it is used
  float x_cur[EPT], x_next[EPT];
  auto fetch_x = [&](int d, int b, float (&dst)[EPT]) {
    const int t0 = (d < n_steps) ? fx_lstm_time(d, 0, T) : -1;
#pragma unroll
    for (int e = 0; e < EPT; ++e) {
      const int k = tid + e * NT;
      dst[e] = (t0 >= 0 && k < HH) ? a.x[((size_t)t0 * B + b) * H + k] : 0.0f;
    }
  };
  fetch_x(0, 0, x_cur);
  int it = 0;   // (step, batch row) pairs so far: its parity picks the buffer of the waves' sums
  for (int d = 0; d < n_steps; ++d) {
    const int rp = (d + 1) & 1;   // parity written by step d - 1
    const uint32_t want = fx_lstm_tag_read(base, d);
    for (int b = 0; b < B; ++b) {
      FX_LSTM_STAMP(0);
      if (b + 1 < B) fetch_x(d, b + 1, x_next);
      else fetch_x(d + 1, 0, x_next);
      // --- element k of what every layer wrote in the step before ---
      // hv[j]: what layer j reads as its own previous h, which is also what layer j + 1 reads as its
      // input: h0[j] at the layer's first step (not tagged), else the h that layer j wrote in step
      // d - 1 (tagged).  A slot that is not tagged or not needed is loaded all the same (and ignored):
      // the loads of a round are then issued together, without a branch and a wait between them, and
      // a round takes one trip to the memory side instead of one per layer.
      bool need[L];
      float hv[L][EPT] = {};
      const uint64_t* src[L];
#pragma unroll
      for (int j = 0; j < L; ++j) {
        const int tj = fx_lstm_time(d, j, T);
        const bool next_active = j + 1 < L && fx_lstm_time(d, j + 1, T) >= 0;
        need[j] = tj != 0 && (tj > 0 || next_active);
        src[j] = a.hbuf + fx_lstm_hoff(rp, j, b, 0, L, B, H);
        if (tj == 0) {
          const float* hr = a.h0 ? a.h0 + ((size_t)j * B + b) * H : nullptr;
#pragma unroll
          for (int e = 0; e < EPT; ++e) hv[j][e] = (hr && tid + e * NT < HH) ? hr[tid + e * NT] : 0.0f;
        }
      }
      {
        uint32_t polls = 0;
        // the waves that are not busy with the cells arrive here while the owners still write: looking
        // at once would only add reads of the very lines the writes are on their way to
        __builtin_amdgcn_s_sleep(FX_LSTM_FIRST_LOOK);
        for (;;) {
          bool ready = true;
          uint64_t el[L][EPT];
#pragma unroll
          for (int j = 0; j < L; ++j)
#pragma unroll
            for (int e = 0; e < EPT; ++e)
              el[j][e] = __hip_atomic_load(src[j] + min(tid + e * NT, HH - 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
          for (int j = 0; j < L; ++j)
#pragma unroll
            for (int e = 0; e < EPT; ++e) {
              ready = ready && (!need[j] || tid + e * NT >= HH || fx_lstm_tag_of(el[j][e]) == want);
              if (need[j]) hv[j][e] = (tid + e * NT < HH) ? __uint_as_float((uint32_t)el[j][e]) : 0.0f;
            }
          if (ready) break;
          if (++polls > a.spin_limit || ((polls & 255u) == 0u && DevAtomics::load(a.ctl + FX_LSTM_W_ERR) != 0u)) {
            // given up (or somebody else has): the workgroup leaves behind this step's barrier
            DevAtomics::store(a.ctl + FX_LSTM_W_ERR, 1u);
            if (a.err_host) __hip_atomic_store(a.err_host, (uint32_t)FX_ASYNC_BARRIER, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            s_abort = 1u;
            break;
          }
          __builtin_amdgcn_s_sleep(1);
        }
      }
      FX_LSTM_STAMP(2);
      // --- this thread's share of every gate sum, and the sums over the wave ---
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        float p[16];   // value (jl * 2 + ul) * 4 + gate
#pragma unroll
        for (int jl = 0; jl < 2; ++jl) {
          const int j = 2 * g + jl;
          const bool active = j < L && fx_lstm_time(d, j < L ? j : 0, T) >= 0;
#pragma unroll
          for (int ul = 0; ul < UPW; ++ul)
#pragma unroll
            for (int gt = 0; gt < 4; ++gt) {
              float s = 0.0f;
              if (j < L) {
#pragma unroll
                for (int e = 0; e < EPT; ++e) {
                  const float in = (j == 0) ? x_cur[e] : hv[j > 0 ? j - 1 : 0][e];
                  s = __builtin_fmaf(w_ih[j < L ? j : 0][gt][ul][e], in, s);
                  s = __builtin_fmaf(w_hh[j < L ? j : 0][gt][ul][e], hv[j < L ? j : 0][e], s);
                }
              }
              p[(jl * 2 + ul) * 4 + gt] = active ? s : 0.0f;
            }
        }
        const float total = wave_sum16(p, lane);   // lane l: the wave's sum of value l >> 2
        if ((lane & 3) == 0) s_part[it & 1][g][wave][lane >> 2] = total;
      }
      FX_LSTM_STAMP(4);
      // the cell states of this batch row, read ahead of the barrier (a lane reads what it wrote itself)
      float c_prev[NG];
#pragma unroll
      for (int g = 0; g < NG; ++g) c_prev[g] = wave == 0 ? s_c[b][(lane & 15) + 16 * g] : 0.0f;
      __syncthreads();
      FX_LSTM_STAMP(5);
      // A wait that was given up: every wave of the workgroup leaves, nothing is checked out.  The
      // first wave looks at the word together with the waves' sums and leaves before it would store.
      if (wave != 0) {
        if (s_abort != 0u) {   // the results are not to be used: the waves without cells say so in the data
          fx_lstm_poison(a, L, (uint32_t)(tid - 64), (uint32_t)(NT - 64));
          return;
        }
      } else {
        // --- sixteen lanes a pair of layers: biases, gates, cells ---
        float part[NG][NW];
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
          for (int w = 0; w < NW; ++w) part[g][w] = s_part[it & 1][g][w][lane & 15];
        const uint32_t aborted = s_abort;
#pragma unroll
        for (int g = 0; g < NG; ++g) {
#pragma unroll
          for (int span = 1; span < NW; span *= 2)
#pragma unroll
            for (int w = 0; w + span < NW; w += 2 * span) part[g][w] += part[g][w + span];
          // the value of a lane here is lane & 15 = (layer in the pair * 2 + unit) * 4 + gate, as for the biases
          const int v = lane & 15, gt = v & 3, ul = (v >> 2) & 1, j = 2 * g + (v >> 3);
          const float pre = (part[g][0] + f_bias_ih[g]) + f_bias_hh[g];
          const float act = gt == 2 ? fx_tanh(pre) : fx_sigmoid(pre);
          const float fg = quad_lane<1>(act), gg = quad_lane<2>(act), og = quad_lane<3>(act);
          const int t = (j < L) ? fx_lstm_time(d, j, T) : -1;
          if (g == 0 && aborted != 0u) return;
          if (lane < 16 && gt == 0 && t >= 0) {
            const float c = (fg * c_prev[g]) + (act * gg);
            s_c[b][lane + 16 * g] = c;
            const float h = og * fx_tanh(c);
            const int u = u0 + ul;
            DevAtomics::store64(a.hbuf + fx_lstm_hoff(d & 1, j, b, u, L, B, H),
                                fx_lstm_pack(__float_as_uint(h), fx_lstm_tag_written(base, d)));
            if (j == L - 1) a.out[((size_t)t * B + b) * H + u] = h;
            if (t == T - 1) {
              a.state_h[((size_t)j * B + b) * H + u] = h;
              a.state_c[((size_t)j * B + b) * H + u] = c;
            }
          }
        }
      }
      FX_LSTM_STAMP(6);
#pragma unroll
      for (int e = 0; e < EPT; ++e) x_cur[e] = x_next[e];
      ++it;
    }
  }
  FX_LSTM_STAMP_END();
  if (threadIdx.x == 0)
    fx_lstm_leave<DevAtomics>(a.ctl, gridDim.x, base, (uint32_t)n_steps, a.hbuf, (uint32_t)(2 * L * B * H));
}

// ---- several sequences at once ----------------------------------------------------------------
// The kernel above walks the batch rows of a step one after the other, and every row pays the whole
// hand-over of its vectors: 2.0 us a row and step, 1 670 us for T = 100, B = 8, H = 256, L = 3.  Here
// a step's products for four rows are one set of matrix instructions and a step costs ONE hand-over.
//   rows     groups of four (v_mfma_f32_4x4x1: tiles of four rows, fp32 in and out).  A group has
//            workgroups of its own, which hold the weights again but wait for, and read, the vectors of
//            their own rows only: what all workgroups read in a step is what the step waits for.
//            H = 512 from nine rows on: two tiles a workgroup, since the device does not hold the
//            workgroups of more groups at once.  (The choice of the form is lstm_forms and what fits.)
//   columns  four hidden units a workgroup.  A vector h_j is multiplied by layer j's recurrent and
//            layer j + 1's input matrix: 16 + 16 gate columns, the 32 columns of a half-wave.
//   depth    the inner dimension is dealt to eight waves in runs of 16: lane l fetches element l / 4
//            of row l % 4 and keeps, in registers for the whole sequence, its column's weights of the
//            eight elements of a run that its half of the wave multiplies (cbsz = 3: a block of four
//            lanes feeds the eight blocks of its half-wave), so a wave sums nothing but its two halves.
//            (Three sizes of H = 512 need more than the 168 registers a lane of a workgroup of this size has
//            and fetch some weights again every step: 6 registers' worth for L = 2 on two tiles, 12 and 52
//            for L = 3 on one and two.  They are no slower than row by row all the same: figures below.)
//   waves    up to four more finish the cells (gate x unit x row: 64 lanes a layer and tile), store
//            them, clear the words of the step after next and bring x into LDS two steps ahead.  A wave
//            that did both would queue its next loads up behind the acknowledgements of its stores.
// Values travel as words (fx_lstm_sched.h): half the bytes of tagged ones.
// T = 100, B = 8, H = 256, L = 3: 273 us, 2.7 us a step, of which 1.6 us pass from the stores to the
// last word seen, 0.25 us are products, 0.7 us cells.  T = 64, H = 512, L = 2: 810 -> 234 us for eight
// rows, 1 620 -> 369 for sixteen, 213 -> 199 for two.
// How long a wave sleeps behind a step's barrier before it first looks at the step's vectors.  A look
// that comes too early costs a whole trip, and its reads slow down the stores they wait for; how long
// the stores take depends on the sizes, so every wave finds its own time: 64 clocks later after an
// early look, 2 clocks sooner after every other one (an early look costs about 30 times 64 clocks).
// T = 100, B = 8, H = 256, L = 3: a fixed 512 clocks 407 us, 1 024: 326, 1 280: 302; this: 277 - 285.
struct FxLook {
  int at = 24 * 32;   // 32nds of 64 clocks
  __device__ __forceinline__ void wait() const {
    for (int n = at >> 5; n > 0; --n) __builtin_amdgcn_s_sleep(1);
  }
  __device__ __forceinline__ void seen(uint32_t polls) { at = polls == 0u ? max(at - 1, 0) : min(at + 32, 64 * 32); }
};
// every store of the wave has been performed at the memory side of the caches
__device__ __forceinline__ void fx_stores_acknowledged() {
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}
// the die that the wave runs on (hardware register XCC_ID, four bits)
__device__ __forceinline__ uint32_t fx_die_of_wave() { return (uint32_t)__builtin_amdgcn_s_getreg(20 | (0 << 6) | (3 << 11)); }
// N consecutive floats of any alignment that floats have
template <int N>
__device__ __forceinline__ void fx_die_load(const float* p, float (&v)[N]) {
  typedef float chunk __attribute__((ext_vector_type(N < 4 ? N : 4), aligned(4)));
#pragma unroll
  for (int i = 0; i < N; i += 4) {
    if constexpr (N == 1) {
      v[0] = *p;
    } else {
      const chunk c = *(const chunk*)(p + i);
#pragma unroll
      for (int k = 0; k < (N < 4 ? N : 4); ++k) v[i + k] = c[k];
    }
  }
}
typedef float fx_f32x4 __attribute__((ext_vector_type(4)));
template <int Q> struct fx_const { static constexpr int value = Q; };
template <class F>
__device__ __forceinline__ void fx_each8(F&& f) {
  f(fx_const<0>()); f(fx_const<1>()); f(fx_const<2>()); f(fx_const<3>());
  f(fx_const<4>()); f(fx_const<5>()); f(fx_const<6>()); f(fx_const<7>());
}

template <int L, int HPT, int MT>
struct FxLstmRows {
  static constexpr int HH = HPT * 32;                   // H
  static constexpr int NW = HPT >= 4 ? 8 : 2 * HPT;     // waves that multiply
  static constexpr int CW = L * MT < 4 ? L * MT : 4;    // waves that finish cells, and bring x
  static constexpr int threads = (NW + CW) * 64;
};
template <int L, int HPT, int MT>
__global__ __launch_bounds__((FxLstmRows<L, HPT, MT>::threads)) void fx_lstm_rows_kernel(const FxLstmArgs a) {
  using C = FxLstmRows<L, HPT, MT>;
  constexpr int HH = C::HH, NW = C::NW, CW = C::CW, NT = C::threads;
  constexpr int KW = HH / NW, KI = KW / 16;             // inner elements of a wave, in runs of 16
  constexpr int S = L + 1;                              // vectors of a step: x and every layer's h
  constexpr int NV = S * MT * 4;                        // partial sums a lane: [vector][tile][row of the tile]
  constexpr int CI = (L * MT + CW - 1) / CW;            // (layer, tile) pairs a wave finishes
  constexpr int XS = HH + 8;                            // distance of x's rows in LDS: the four rows a wave reads lie in different banks
  constexpr int XP = (MT * HH + CW * 64 - 1) / (CW * 64);   // 16-byte groups of x a lane brings in
  __shared__ float s_part[2][NW][NV * 32];              // by parity of the step: [(vector, tile)][column half][row][16]
  __shared__ float s_x[3][4 * MT * XS];                 // x of a step and of the two behind it
  __shared__ uint32_t s_abort;
  FX_LSTM_STAMP_DECL
  const int B = a.B, T = a.T;
  const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
  constexpr int n_wg = HH / 4;                          // workgroups of a group of rows
  const int group = (int)blockIdx.x / n_wg, gi = (int)blockIdx.x % n_wg;
  // as above: the workgroups of a die take neighbouring hidden units
  const int wg = (n_wg % 8 == 0) ? (gi % 8) * (n_wg / 8) + gi / 8 : gi;
  const int u0 = wg * 4;
  const int b0 = group * 4 * MT, nb = min(4 * MT, B - b0);
  if (tid == 0) s_abort = fx_lstm_refused<DevAtomics>(a) ? 1u : 0u;
  const uint32_t base = DevAtomics::load(a.ctl + FX_LSTM_W_BASE);
  const int n_steps = fx_lstm_steps(T, L);
  const uint32_t BH = (uint32_t)(B * HH);               // elements of one vector of all rows
  const int c_ul = (lane >> 2) & 3, c_gate = lane & 3;

  if (wave < NW) {
    // ---- products.  This lane's column: lanes 0-15 of a half-wave the recurrent matrix of the vector's own
    // layer, lanes 16-31 the input matrix of the layer above; unit (lane >> 2) & 3, gate lane & 3.
    // Element of a wave's run that block `blk` (four lanes) fetches: pairs of neighbours where there is a
    // second run.
    const int half = (lane >> 4) & 1;
    auto k_of = [&](int i, int blk) { return wave * KW + (KI == 1 ? blk : 32 * (i / 2) + 2 * blk + (i & 1)); };
    float w[S][KI][8];
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const int jc = half ? s : s - 1;                  // the layer whose gates the column belongs to
      const bool live = jc >= 0 && jc < L;              // (x has no recurrent matrix, the last h no layer above)
      const int j = min(max(jc, 0), L - 1);
      const float* m = half ? a.wih : a.whh;
#pragma unroll
      for (int i = 0; i < KI; ++i)
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const float v = m[((size_t)(j * 4 + c_gate) * HH + k_of(i, 8 * (lane >> 5) + q)) * HH + u0 + c_ul];
          w[s][i][q] = live ? v : 0.0f;
        }
    }
    // word (row, k) of a vector that this lane fetches, per tile; rows past the batch repeat its last one
    // (their sums are not used)
    uint32_t at[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) at[mt] = (uint32_t)((b0 + min(mt * 4 + (lane & 3), nb - 1)) * HH + k_of(0, lane >> 2));
    const int xat = (lane & 3) * XS + k_of(0, lane >> 2);
    __syncthreads();
    if (s_abort != 0u) {   // uniform: written once, ahead of the barrier
      if (tid == 0 && a.err_host) __hip_atomic_store(a.err_host, (uint32_t)FX_ASYNC_BARRIER, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      fx_lstm_poison(a, L, (uint32_t)tid, (uint32_t)(NW * 64));
      return;
    }
    FxLook look;
    for (int d = 0; d < n_steps; ++d) {
      FX_LSTM_STAMP(0);
      fx_f32x4 acc[S][MT];
#pragma unroll
      for (int s = 0; s < S; ++s)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[s][mt] = fx_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      // one matrix instruction: element 8 * (half-wave) + Q of a run, for every column of a vector.  Its
      // callers go round the vectors before they come back to an accumulator: a dependent one waits.
      auto multiply = [&](auto q, int s, int mt, int i, float v) {
        constexpr int Q = decltype(q)::value;
        acc[s][mt] = __builtin_amdgcn_mfma_f32_4x4x1f32(v, w[s][i][Q], acc[s][mt], 3, Q, 0);
      };
      // x is known ahead: its products fill the time in which the other workgroups' values travel
      {
        float xv[MT][KI];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int i = 0; i < KI; ++i) xv[mt][i] = s_x[d % 3][mt * 4 * XS + xat + (KI == 1 ? 0 : 32 * (i / 2) + (i & 1))];
#pragma unroll
        for (int i = 0; i < KI; ++i)
          fx_each8([&](auto q) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) multiply(q, 0, mt, i, xv[mt][i]);
          });
      }
      FX_LSTM_STAMP(1);
      // the h vectors, as above: words of the step before, h0 at a layer's first step
      float hv[L][MT][KI];
      bool need[L];
#pragma unroll
      for (int j = 0; j < L; ++j) {
        const int tj = fx_lstm_time(d, j, T);
        need[j] = tj != 0 && (tj > 0 || (j + 1 < L && fx_lstm_time(d, j + 1, T) >= 0));
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int i = 0; i < KI; ++i)
            hv[j][mt][i] = (tj == 0 && a.h0) ? (a.h0 + (size_t)j * BH)[at[mt] + (KI == 1 ? 0 : 32 * (i / 2) + (i & 1))] : 0.0f;
      }
      const uint32_t* src = (const uint32_t*)a.hbuf + (size_t)fx_lstm_slot(base, d - 1) * (L * BH);
      uint32_t polls = 0;
      if (d > 0) look.wait();
      for (;;) {
        bool ready = true;
        uint32_t el[L][MT][KI];
#pragma unroll
        for (int j = 0; j < L; ++j)
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) {
            if constexpr (KI == 1) {
              el[j][mt][0] = __hip_atomic_load(src + (size_t)j * BH + at[mt], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            } else {
#pragma unroll
              for (int i = 0; i < KI; i += 2) {
                const uint64_t two = __hip_atomic_load((const uint64_t*)(src + (size_t)j * BH + at[mt] + 16 * i), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                el[j][mt][i] = (uint32_t)two;
                el[j][mt][i + 1] = (uint32_t)(two >> 32);
              }
            }
          }
#pragma unroll
        for (int j = 0; j < L; ++j)
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int i = 0; i < KI; ++i) {
              ready = ready && (!need[j] || el[j][mt][i] != 0u);
              hv[j][mt][i] = need[j] ? __uint_as_float(fx_lstm_word_value(el[j][mt][i])) : hv[j][mt][i];
            }
        if (!wave_any(!ready)) break;   // (a matrix instruction reads its operands from all lanes)
        if (++polls > a.spin_limit || ((polls & 255u) == 0u && DevAtomics::load(a.ctl + FX_LSTM_W_ERR) != 0u)) {
          // given up (or somebody else has): the workgroup leaves behind this step's barrier
          DevAtomics::store(a.ctl + FX_LSTM_W_ERR, 1u);
          if (a.err_host) __hip_atomic_store(a.err_host, (uint32_t)FX_ASYNC_BARRIER, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
          s_abort = 1u;
          break;
        }
      }
      look.seen(polls);
      FX_LSTM_POLLS(polls);
      FX_LSTM_STAMP(2);
#pragma unroll
      for (int i = 0; i < KI; ++i)
        fx_each8([&](auto q) {
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int j = 0; j < L; ++j) multiply(q, j + 1, mt, i, hv[j][mt][i]);
        });
      FX_LSTM_STAMP(3);
      // the two halves of the wave: the lower keeps the first half of the values, the upper the second
      float* dst = s_part[d & 1][wave];
#pragma unroll
      for (int i = 0; i < NV / 2; ++i) {
        const float lo = acc[(i >> 2) / MT][(i >> 2) % MT][i & 3];
        const float hi = acc[((i + NV / 2) >> 2) / MT][((i + NV / 2) >> 2) % MT][(i + NV / 2) & 3];
        const fx_u32x2v t = __builtin_amdgcn_permlane32_swap(__float_as_uint(lo), __float_as_uint(hi), false, false);
        const int v = i + (lane >> 5) * (NV / 2);
        dst[(((v >> 2) * 2 + half) * 4 + (v & 3)) * 16 + (lane & 15)] = __uint_as_float(t.x) + __uint_as_float(t.y);
      }
      FX_LSTM_STAMP(4);
      __syncthreads();
      FX_LSTM_STAMP(5);
      if (s_abort != 0u) {   // the results are not to be used: say so in the data
        fx_lstm_poison(a, L, (uint32_t)tid, (uint32_t)(NW * 64));
        return;
      }
    }
    FX_LSTM_STAMP_END();
    __syncthreads();   // the last step's values
    return;
  }

  // ---- cells: lane = row of the tile * 16 + unit * 4 + gate; pair jt = layer * MT + tile ----
  const int cw = wave - NW, f_m = lane >> 4;
  float bias_ih[CI], bias_hh[CI], cell[CI];
#pragma unroll
  for (int ci = 0; ci < CI; ++ci) {
    const int jt = min(cw + CW * ci, L * MT - 1), j = jt / MT, b = b0 + min((jt % MT) * 4 + f_m, nb - 1);
    bias_ih[ci] = a.bih[(size_t)(j * 4 + c_gate) * HH + u0 + c_ul];
    bias_hh[ci] = a.bhh[(size_t)(j * 4 + c_gate) * HH + u0 + c_ul];
    cell[ci] = a.c0 ? a.c0[((size_t)j * B + b) * HH + u0 + c_ul] : 0.0f;
  }
  fx_u32x4_a4 xr[XP];
  auto fetch_x = [&](int d) {   // (unconditional: what a step without its first layer reads is not used)
    const float* src = a.x + (size_t)min(d, T - 1) * BH;
#pragma unroll
    for (int e = 0; e < XP; ++e) {
      const int g = min(cw * 64 + lane + CW * 64 * e, MT * HH - 1), r = g / (HH / 4), c = g % (HH / 4);
      xr[e] = *(const fx_u32x4_a4*)(src + (size_t)(b0 + min(r, nb - 1)) * HH + 4 * c);
    }
  };
  auto park_x = [&](int d) {
#pragma unroll
    for (int e = 0; e < XP; ++e) {
      const int g = min(cw * 64 + lane + CW * 64 * e, MT * HH - 1), r = g / (HH / 4), c = g % (HH / 4);
      *(fx_u32x4*)(s_x[d % 3] + r * XS + 4 * c) = xr[e];
    }
  };
  fetch_x(0);
  park_x(0);
  fetch_x(1);
  park_x(1);
  fetch_x(2);
  __syncthreads();
  if (s_abort != 0u) return;
  for (int d = 0; d < n_steps; ++d) {
    __syncthreads();
    FX_LSTM_STAMP(5);
    const uint32_t aborted = s_abort;
    const uint32_t out_slot = fx_lstm_slot(base, d) * (uint32_t)(L * BH), clear_slot = fx_lstm_slot(base, d + 2) * (uint32_t)(L * BH);
    if (aborted != 0u) return;   // uniform, ahead of every store of the step
#pragma unroll
    for (int ci = 0; ci < CI; ++ci) {
      const int jt = cw + CW * ci, j = jt / MT, mt = jt % MT;
      const int t = jt < L * MT ? fx_lstm_time(d, j, T) : -1;
      if (t < 0) continue;   // uniform in the wave
      float ih[NW], hh[NW];
#pragma unroll
      for (int g = 0; g < NW; ++g) {
        ih[g] = s_part[d & 1][g][((j * MT + mt) * 2 + 1) * 64 + lane];
        hh[g] = s_part[d & 1][g][(((j + 1) * MT + mt) * 2) * 64 + lane];
      }
#pragma unroll
      for (int g = 0; g < NW; ++g) ih[g] += hh[g];
#pragma unroll
      for (int span = 1; span < NW; span *= 2)
#pragma unroll
        for (int g = 0; g + span < NW; g += 2 * span) ih[g] += ih[g + span];
      const float pre = (ih[0] + bias_ih[ci]) + bias_hh[ci];
      const float act = c_gate == 2 ? fx_tanh(pre) : fx_sigmoid(pre);
      const float fg = quad_lane<1>(act), gg = quad_lane<2>(act), og = quad_lane<3>(act);
      const int r = mt * 4 + f_m;
      if (c_gate == 0 && r < nb) {
        const float c = (fg * cell[ci]) + (act * gg);
        cell[ci] = c;
        const float h = og * fx_tanh(c);
        const int b = b0 + r, u = u0 + c_ul;
        DevAtomics::store((uint32_t*)a.hbuf + out_slot + (uint32_t)((j * B + b) * HH + u), fx_lstm_word(__float_as_uint(h)));
        if (j == L - 1) a.out[((size_t)t * B + b) * HH + u] = h;
        if (t == T - 1) {
          a.state_h[((size_t)j * B + b) * HH + u] = h;
          a.state_c[((size_t)j * B + b) * HH + u] = c;
        }
      }
    }
    FX_LSTM_STAMP(6);
    // between the barriers of steps d and d + 1 the others read x of step d + 1; the slot of step d + 2
    // was last read in step d - 1
    park_x(d + 2);
#pragma unroll
    for (int ci = 0; ci < CI; ++ci) {
      const int jt = cw + CW * ci, r = (jt % MT) * 4 + f_m;
      if (jt < L * MT && c_gate == 0 && r < nb)
        DevAtomics::store((uint32_t*)a.hbuf + clear_slot + (uint32_t)(((jt / MT) * B + b0 + r) * HH + u0 + c_ul), 0u);
    }
    fx_stores_acknowledged();   // ahead of the next barrier (the others are busy until then)
    fetch_x(d + 3);
    FX_LSTM_STAMP(7);
  }
  FX_LSTM_STAMP_END();
  __syncthreads();   // every wave's values are at the memory side before the workgroup checks out
  if (cw == 0 && lane == 0) fx_lstm_leave_slots<DevAtomics>(a.ctl, gridDim.x, base, (uint32_t)n_steps);
}

// ---- a sequence on one die ---------------------------------------------------------------------
// What the kernels above spend most of a step on is the hand-over: a value goes to the memory side of the
// caches and comes back from there, 0.45 us one way at its quickest and 0.9 to 1.6 with every workgroup of the
// chip reading.  The compute units of one die share a cache: a store that stays in it is seen by a load of
// another unit after 0.2 us.  A die's registers hold the weights of one layer of 512 units, or of all layers
// of fewer, so here a sequence's layers (a stage of them, fx_lstm_sched.h) run on the 32 units of a die and
// sequences on dies of their own; only h between stages crosses, and nothing waits for that.
//   columns  a workgroup has 2 E of the 64 E hidden units, 8 E gate columns a layer.
//   depth    dealt to eight waves in runs of 8 E.  Lane (kl, cl) = (lane >> 3, lane & 7) multiplies E elements
//            by E columns: gate cl >> 1 of E units.  A lane fetches ONE element and has the others of its
//            group of E lanes by lane-crossing moves; sums are taken over kl only.
//   shadow   the products with the layer's input (x, or h of the layer below, two steps old) come first: they
//            fill the time in which the layer's own h travels.
//   cells    one or two more waves: a lane a gate column, four lanes a cell; they bring the stage's input into
//            LDS two steps ahead.
// Where a workgroup runs is the hardware's choice (dies in turn).  Loads are device-scope either way; whether a
// value may be stored to the die's cache only, the workgroups of a stage find out while they load their
// weights: each publishes its die, and unless all agree they store to the memory side.
// That a value stored at workgroup scope is seen by a device-scope load of another unit of the die is how this chip
// is built (first-level caches write through; device-scope loads pass them and find what lies in the die's cache,
// written back or not), not what the memory model promises: between workgroups it is relied on only where the die is the same.
// us a launch, T = 64, this : the forms above: 512 units, one sequence, one to three layers 80 : 110, 92 : 119, 98 : 188;
// two layers, four sequences 98 : 219; 256 units, four layers, four sequences 89 : 207; 128, three, eight 71 : 125;
// 64, one, one 47 : 105.  T = 100, 256 units, three layers, eight sequences 131 : 269.  T = 8: 27 : 28 (512, two
// layers), 12 : 16 (64, one); shorter sequences: fx_lstm_die_from.
// The same workgroups spread over the chip (spread: slot after slot, every slot on all dies; only those that have a
// sequence are launched) compute the same bits with values that go to the memory side, for launches that must
// not hold a die: 512 units, two layers, one sequence 93 on dies, 101 spread (110 before neighbouring units were one die's), 119 row
// by row; three layers of 256, four sequences 91, 111, 178 (tiles of rows); 128, three, eight 70, 102, 125; 64, three, eight 60, 94, 106;
// 64, one, one 46, 73, 106.
// A step of two layers of 512 units is 1.1 us:
// 0.3 from the barrier to the cells' stores, 0.3 until they are seen, 0.35 products, 0.1 sums (on the SIMD that also
// finishes cells, the others wait for it); of 64 units 0.65.
template <int CTRL>
__device__ __forceinline__ float fx_dpp(float v) { return dpp_get<CTRL>(v); }
// element e of the lane's group of E lanes; E = 8: the upper four in mirrored order (fx_die_element)
template <int E>
__device__ __forceinline__ void fx_die_spread(float h, float (&v)[E]) {
  if constexpr (E == 1) v[0] = h;
  if constexpr (E == 2) {
    v[0] = fx_dpp<0xA0>(h);   // quad_perm [0, 0, 2, 2]
    v[1] = fx_dpp<0xF5>(h);   // quad_perm [1, 1, 3, 3]
  }
  if constexpr (E >= 4) {
    v[0] = quad_lane<0>(h); v[1] = quad_lane<1>(h); v[2] = quad_lane<2>(h); v[3] = quad_lane<3>(h);
  }
  if constexpr (E == 8) {
    const float m = fx_dpp<0x141>(h);   // row_half_mirror: the other four of the group
    v[4] = quad_lane<0>(m); v[5] = quad_lane<1>(m); v[6] = quad_lane<2>(m); v[7] = quad_lane<3>(m);
  }
}
template <int E>
__device__ __forceinline__ int fx_die_element(int cl, int e) {   // which element of the group spread's v[e] is
  return E < 8 ? e : e < 4 ? 4 * (cl >> 2) + e : 11 - 4 * (cl >> 2) - e;
}
// V values a lane, summed over the lanes that differ in bits 3, 4 and 5 of their number; where the count is even
// a stage keeps half of the values in each lane.  Left: fx_die_left(V) values from *first on.
constexpr int fx_die_left(int v) {
  for (int i = 0; i < 3; ++i) v = v % 2 == 0 ? v / 2 : v;
  return v;
}
template <int V, int BIT>
__device__ __forceinline__ void fx_die_sum(float (&p)[V], int lane, int* first, float* out) {
  constexpr bool halve = V % 2 == 0;
  constexpr int N = halve ? V / 2 : V;
  float q[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const float a = p[i], b = halve ? p[(i + N) % V] : p[i];
    if constexpr (BIT == 3) {
      const bool up = halve && (lane & 8) != 0;
      const float keep = up ? b : a, send = up ? a : b;
      q[i] = keep + fx_dpp<0x128>(send);   // row_ror:8: from lane l ^ 8
    } else {
      const fx_u32x2v t = BIT == 5 ? __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false)
                                   : __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
      q[i] = __uint_as_float(t.x) + __uint_as_float(t.y);
    }
  }
  if (halve) *first += ((lane >> BIT) & 1) * N;
  if constexpr (BIT > 3) {
    fx_die_sum<N, BIT - 1>(q, lane, first, out);
  } else {
#pragma unroll
    for (int i = 0; i < N; ++i) out[i] = q[i];
  }
}

// The activation of a gate: tanh for the cell gate, sigmoid for the others, by way of one exponential
// (fx_sigmoid's; lanes of both kinds are in one wave, which would go through two).
__device__ __forceinline__ float fx_die_gate(float x, bool cell_gate) {
  const float l2e_hi = 1.44269502e+00f, l2e_lo = 1.92596299e-08f, ln2 = 6.93147182e-01f;
  const float ax = fabsf(x), arg = cell_gate ? 2.0f * ax : -x;
  const float th = arg * l2e_hi;
  const float tl = __builtin_fmaf(arg, l2e_hi, -th) + arg * l2e_lo;
  float e = __builtin_amdgcn_exp2f(th);
  e = __builtin_fmaf(e, tl * ln2, e);
  float r = __builtin_amdgcn_rcpf(1.0f + e);
  r = (th > 128.0f) ? 0.0f : r;
  r = (th < -150.0f) ? 1.0f : r;
  const float z = x * x;   // as fx_tanh: a polynomial where 1 - 2 r would cancel
  float p = -5.70498872745e-3f;
  p = __builtin_fmaf(p, z, 2.06390887954e-2f);
  p = __builtin_fmaf(p, z, -5.37397155531e-2f);
  p = __builtin_fmaf(p, z, 1.33314422036e-1f);
  p = __builtin_fmaf(p, z, -3.33332819422e-1f);
  const float small = __builtin_fmaf(p * z, x, x);
  const float t = ax < 0.625f ? small : copysignf(1.0f - 2.0f * r, x);
  return cell_gate ? t : r;
}

template <int E, int NL>
struct FxLstmDie {
  static constexpr int HH = 64 * E, C = 8 * E, U = 2 * E;   // units; gate columns a layer and units of a workgroup
  static constexpr int NW = 8, CW = (NL * C + 63) / 64;     // waves that multiply, waves that finish cells
  static constexpr int threads = (NW + CW) * 64;
  // Units of 64 clocks that a wave sleeps ahead of its first look: values are there some 1 100 clocks behind the
  // barrier, and looks slow down the stores that they wait for.  Longer products are long enough.  (One layer of 64
  // units, T = 64: 0 to 4 units 52 us, 6 48, 8 46.7, 9 47; 128 units: 2 to 9 within 4 %.)
  static constexpr int sleep = E == 1 ? 9 - NL : E == 2 ? 2 : E * NL == 4 ? 1 : 0;
  // The same where the workgroups are spread over the dies and a value takes a microsecond (T = 64, units : us.  64 units, one
  // layer: 0 129, 8 98, 16 77, 24 85; 128, three layers, eight sequences: 0 147, 16 101; 256, three, four: 0 134, 14 114;
  // 512, two, one: 0 112, 8 110, 16 120)
  static constexpr int sleep_spread = E == 1 ? 16 : E == 2 ? 15 : E == 4 ? 14 : 8;
};
template <int E, int NL>
__global__ __launch_bounds__((FxLstmDie<E, NL>::threads)) void fx_lstm_die_kernel(const FxLstmArgs a, int L, int spread) {
  using K = FxLstmDie<E, NL>;
  constexpr int HH = K::HH, C = K::C, NW = K::NW, NC = NL * C;
  __shared__ float s_part[2][NW][NC];   // the waves' sums, by parity of the step: [layer][unit][gate]
  __shared__ __align__(16) float s_in[3][HH];   // the stage's input of a step and of the two behind it
  // A wait that is given up between the barriers of steps d - 1 and d sets word d & 1, which is read behind barrier d
  // and not set again before barrier d + 1: all waves of the workgroup see the same and leave at the same place.
  // (Ahead of step 0's barrier there is one more, of step -1.)
  __shared__ uint32_t s_abort[2];
  const int B = a.B, T = a.T;
  const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int slot = spread ? (int)blockIdx.x / FX_LSTM_DIE_WG : (int)blockIdx.x % FX_LSTM_DIES;
  // (spread: workgroups of one die, every eighth, take neighbouring units, whose weights share lines)
  const int gi = spread ? ((int)blockIdx.x % FX_LSTM_DIES) * (FX_LSTM_DIE_WG / FX_LSTM_DIES) + (int)blockIdx.x % FX_LSTM_DIE_WG / FX_LSTM_DIES
                        : (int)blockIdx.x / FX_LSTM_DIES;
  const int stages = L / NL, b = slot / stages, stage = slot % stages, j0 = stage * NL;
  const int u0 = gi * K::U;
  const int n_steps = fx_lstm_stage_steps(T, NL);
  const uint32_t advance = (uint32_t)n_steps + 1u;   // tags that a launch uses
  const FxLstmDieArea area = fx_lstm_die_area(B, HH, L);
  const uint32_t parity = (uint32_t)(L * B * HH);   // from one half of the h buffer to the other
  const uint32_t base = DevAtomics::load(a.ctl + FX_LSTM_W_BASE);
  if (b >= B) {   // no sequence for this die
    if (tid == 0) fx_lstm_leave<DevAtomics>(a.ctl, gridDim.x, base, advance, a.hbuf, area.words);
    return;
  }
  if (tid < 2) s_abort[tid] = 0u;
  __syncthreads();
  if (tid == 0 && fx_lstm_refused<DevAtomics>(a)) s_abort[1] = 1u;
  uint64_t* const where = a.hbuf + area.where + slot * FX_LSTM_DIE_WG;
  if (tid == 0) DevAtomics::store64(where + gi, fx_lstm_pack(fx_die_of_wave(), base + 1u));
  auto give_up = [&](int d) {   // the workgroup leaves behind the barrier of step d, the next one
    DevAtomics::store(a.ctl + FX_LSTM_W_ERR, 1u);
    if (a.err_host) __hip_atomic_store(a.err_host, (uint32_t)FX_ASYNC_BARRIER, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    s_abort[d & 1] = 1u;
  };
  // polls so far of a wait: is it to be given up?
  auto too_long = [&](uint32_t polls) {
    return polls > a.spin_limit || ((polls & 255u) == 0u && DevAtomics::load(a.ctl + FX_LSTM_W_ERR) != 0u);
  };

  if (wave < NW) {
    const int kl = lane >> 3, cl = lane & 7;
    float w_ih[NL][E][E], w_hh[NL][E][E];   // [layer][element][column]
#pragma unroll
    for (int k = 0; k < NL; ++k)
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const size_t at = ((size_t)((j0 + k) * 4 + (cl >> 1)) * HH + wave * 8 * E + kl * E + fx_die_element<E>(cl, e)) * HH + u0 + (cl & 1) * E;
        fx_die_load<E>(a.wih + at, w_ih[k][e]);
        fx_die_load<E>(a.whh + at, w_hh[k][e]);
      }
    const int own = wave * 8 * E + kl * E + cl % E;   // the element that this lane fetches
    float below[NL] = {};                              // h of the layer below, read in the step before
    const uint64_t* from[NL];
#pragma unroll
    for (int k = 0; k < NL; ++k) from[k] = a.hbuf + fx_lstm_hoff(0, j0 + k, b, own, L, B, HH);
    __builtin_amdgcn_s_waitcnt(0);   // (the weights are here: otherwise the loop waits for them, and for looks behind them)
    __syncthreads();
    if (s_abort[1] != 0u) {
      if (tid == 0 && a.err_host) __hip_atomic_store(a.err_host, (uint32_t)FX_ASYNC_BARRIER, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      fx_lstm_poison(a, L, (uint32_t)tid, (uint32_t)(NW * 64));
      return;
    }
    // Step d; all: every layer is in the middle of the sequence, and nothing is asked about one.
    // What this lane's products are multiplied by comes through s_in[place] and from the die's cache.
    uint32_t aborted = 0u;
    auto step = [&](auto every, int d, int place) {
      constexpr bool all = decltype(every)::value != 0;
      float acc[NL * E];
#pragma unroll
      for (int i = 0; i < NL * E; ++i) acc[i] = 0.0f;
      // Sums of E = 8: chains of four products, added up in a tree.  A chain of sixteen loses what the sums over the
      // lanes keep (T = 64, 512 units, two layers, mean of eight inputs against 64 bits: 2.11e-7; so 1.83e-7, row by row
      // 1.86e-7).
      auto multiply = [&](float h, const float (&w)[E][E], int k) {
        float v[E];
        fx_die_spread<E>(h, v);
        if constexpr (E < 8) {
#pragma unroll
          for (int e = 0; e < E; ++e)
#pragma unroll
            for (int c = 0; c < E; ++c) acc[k * E + c] = __builtin_fmaf(w[e][c], v[e], acc[k * E + c]);
        } else {
          float sum[2][E];
#pragma unroll
          for (int e = 0; e < E; ++e)
#pragma unroll
            for (int c = 0; c < E; ++c) sum[e / 4][c] = e % 4 == 0 ? w[e][c] * v[e] : __builtin_fmaf(w[e][c], v[e], sum[e / 4][c]);
#pragma unroll
          for (int c = 0; c < E; ++c) acc[k * E + c] += sum[0][c] + sum[1][c];
        }
      };
#pragma unroll
      for (int k = 0; k < NL; ++k)
        if (all || fx_lstm_stage_time(d, k, T) >= 0) multiply(k == 0 ? s_in[place][own] : below[k > 0 ? k - 1 : 0], w_ih[k], k);
#pragma unroll
      for (int i = 0; i < NL * E; ++i) asm volatile("" : "+v"(acc[i]));   // (they are not to sink behind the wait)
      if (aborted != 0u) return;   // uniform
      bool need[NL];
      float hv[NL];
#pragma unroll
      for (int k = 0; k < NL; ++k) {
        const int t = all ? 1 : fx_lstm_stage_time(d, k, T);
        need[k] = all || (d > 0 && fx_lstm_stage_time(d - 1, k, T) >= 0 && (t >= 0 || k + 1 < NL));
        hv[k] = !all && t == 0 && a.h0 ? a.h0[((size_t)(j0 + k) * B + b) * HH + own] : 0.0f;
      }
      const uint32_t want = fx_lstm_tag_read(base, d);
      if (spread) __builtin_amdgcn_s_sleep(K::sleep_spread);
      else if constexpr (K::sleep > 0) __builtin_amdgcn_s_sleep(K::sleep);
      for (uint32_t polls = 0;;) {
        uint64_t el[NL];
        bool ready = true;
#pragma unroll
        for (int k = 0; k < NL; ++k)
          el[k] = __hip_atomic_load(from[k] + ((d + 1) & 1) * parity, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int k = 0; k < NL; ++k) ready = ready && (!need[k] || fx_lstm_tag_of(el[k]) == want);
#pragma unroll
        for (int k = 0; k < NL; ++k) hv[k] = need[k] ? __uint_as_float((uint32_t)el[k]) : hv[k];
        if (!wave_any(!ready)) break;
        if (too_long(++polls)) {
          give_up(d);
          break;
        }
      }
#pragma unroll
      for (int k = 0; k < NL; ++k) {
        if (all || fx_lstm_stage_time(d, k, T) >= 0) multiply(hv[k], w_hh[k], k);
        below[k] = hv[k];
      }
      constexpr int left = fx_die_left(NL * E);
      int first = 0;
      float sum[left];
      fx_die_sum<NL * E, 5>(acc, lane, &first, sum);
#pragma unroll
      for (int i = 0; i < left; ++i) {
        const int v = first + i, k = v / E, unit = (cl & 1) * E + v % E;
        s_part[d & 1][wave][k * C + unit * 4 + (cl >> 1)] = sum[i];
      }
      __syncthreads();
      aborted = s_abort[d & 1];   // (looked at behind the next products)
    };
    int place = 0;
    for (int d = 0; d < n_steps && aborted == 0u; ++d) {
      if (d > 2 * (NL - 1) && d < T) step(fx_const<1>(), d, place);
      else step(fx_const<0>(), d, place);
      place = place == 2 ? 0 : place + 1;
    }
    if (aborted != 0u) {   // the results are not to be used: say so in the data
      fx_lstm_poison(a, L, (uint32_t)tid, (uint32_t)(NW * 64));
      return;
    }
    __syncthreads();   // the last step's values
    return;
  }

  // ---- cells: lane f = (layer of the stage, unit, gate) ----
  const int cw = wave - NW, f = min(cw * 64 + lane, NC - 1), fk = f / C, gate = f & 3, u = u0 + ((f % C) >> 2), j = j0 + fk;
  const float bias_ih = a.bih[(size_t)(j * 4 + gate) * HH + u], bias_hh = a.bhh[(size_t)(j * 4 + gate) * HH + u];
  float cell = a.c0 ? a.c0[((size_t)j * B + b) * HH + u] : 0.0f;
  __builtin_amdgcn_s_setprio(3);   // (the waves that multiply share the SIMDs: ahead of them)
  const bool owner = gate == 0 && cw * 64 + lane < NC;
  const bool last = fk == NL - 1;
  uint64_t* const h_to = a.hbuf + fx_lstm_hoff(0, j, b, u, L, B, HH);
  // the stage's input: x, or what the stage before puts into its ring
  const int link = (stage - 1) * B + b;
  const uint64_t* const ring_in = a.hbuf + area.ring + (size_t)(link < 0 ? 0 : link) * (FX_LSTM_RING * HH);
  uint64_t* const ring_out = a.hbuf + area.ring + (size_t)(stage * B + b) * (FX_LSTM_RING * HH);
  uint64_t* const read_in = a.hbuf + area.read + (link < 0 ? 0 : link) * FX_LSTM_DIE_WG + gi;
  const uint64_t* const read_out = a.hbuf + area.read + (stage * B + b) * FX_LSTM_DIE_WG;
  float in[E];
  auto fetch = [&](int t) {   // x of step t, asked for
    if (stage == 0 && t < T) fx_die_load<E>(a.x + ((size_t)t * B + b) * HH + lane * E, in);
  };
  auto park = [&](int t, int d) {   // d: whose barrier is next
    if (t >= T) return;
    if (stage > 0) {
      for (uint32_t polls = 0;;) {
        bool ready = true;
#pragma unroll
        for (int e = 0; e < E; ++e) {
          const uint64_t el = __hip_atomic_load(ring_in + (t % FX_LSTM_RING) * HH + e * 64 + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          ready = ready && fx_lstm_tag_of(el) == base + (uint32_t)t + 1u;
          in[e] = __uint_as_float((uint32_t)el);
        }
        if (!wave_any(!ready)) break;
        if (too_long(++polls)) {
          give_up(d);
          break;
        }
      }
      if (lane == 0) DevAtomics::store64(read_in, (uint64_t)(base + (uint32_t)t + 1u));
#pragma unroll
      for (int e = 0; e < E; ++e) s_in[t % 3][e * 64 + lane] = in[e];
    } else {
#pragma unroll
      for (int e = 0; e < E; ++e) s_in[t % 3][lane * E + e] = in[e];
    }
  };
  bool same_die = true;
  for (uint32_t polls = 0;;) {
    const uint64_t el = __hip_atomic_load(where + (lane & (FX_LSTM_DIE_WG - 1)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (!wave_any(fx_lstm_tag_of(el) != base + 1u)) {
      same_die = !wave_any((uint32_t)el != fx_die_of_wave());
      break;
    }
    if (too_long(++polls)) {
      give_up(-1);
      break;
    }
  }
  if (cw == 0) {
    for (int t = 0; t < 2; ++t) {
      fetch(t);
      park(t, -1);
    }
    fetch(2);
  }
  __syncthreads();
  if (s_abort[1] != 0u) return;
  for (int d = 0; d < n_steps; ++d) {
    __syncthreads();
    const uint32_t aborted = s_abort[d & 1];
    float part[NW];
#pragma unroll
    for (int w = 0; w < NW; ++w) part[w] = s_part[d & 1][w][f];
#pragma unroll
    for (int span = 1; span < NW; span *= 2)
#pragma unroll
      for (int w = 0; w + span < NW; w += 2 * span) part[w] += part[w + span];
    const float pre = (part[0] + bias_ih) + bias_hh;
    const float act = fx_die_gate(pre, gate == 2);
    const float fg = quad_lane<1>(act), gg = quad_lane<2>(act), og = quad_lane<3>(act);
    const int t = fx_lstm_stage_time(d, fk, T);
    if (owner && t >= 0 && aborted == 0u) {
      cell = (fg * cell) + (act * gg);
      const float h = og * fx_tanh(cell);
      uint64_t* const to = h_to + (d & 1) * parity;
      const uint64_t el = fx_lstm_pack(__float_as_uint(h), fx_lstm_tag_written(base, d));
      if (same_die) __hip_atomic_store(to, el, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      else DevAtomics::store64(to, el);
      if (last && stage + 1 < stages) DevAtomics::store64(ring_out + (t % FX_LSTM_RING) * HH + u, fx_lstm_pack(__float_as_uint(h), base + (uint32_t)t + 1u));
      if (j == L - 1) a.out[((size_t)t * B + b) * HH + u] = h;
      if (t == T - 1) {
        a.state_h[((size_t)j * B + b) * HH + u] = h;
        a.state_c[((size_t)j * B + b) * HH + u] = cell;
      }
    }
    if (aborted != 0u) return;   // uniform, and nothing of this step was stored
    // between the barriers of steps d and d + 1 the others read the input of step d + 1; the place of step
    // d + 2 was last read in step d - 1
    if (cw == 0) {
      park(d + 2, d + 1);
      fetch(d + 3);
    }
    // every half ring: the next half may be written (the next stage is never that far behind but at the start)
    if (stage + 1 < stages && d + 1 < n_steps && d % (FX_LSTM_RING / 2) == FX_LSTM_RING / 2 - 1) {
      const int seen = d + 1 - FX_LSTM_RING / 2;   // vectors that have to be read before vector d + RING / 2 is written
      for (uint32_t polls = 0; seen > 0;) {
        const uint32_t n = (uint32_t)__hip_atomic_load(read_out + (lane & (FX_LSTM_DIE_WG - 1)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (!wave_any((int32_t)(n - (base + (uint32_t)seen)) < 0)) break;
        if (too_long(++polls)) {
          give_up(d + 1);
          break;
        }
      }
    }
  }
  __syncthreads();   // the waves that multiply are done
  if (cw == 0 && lane == 0) fx_lstm_leave<DevAtomics>(a.ctl, gridDim.x, base, advance, a.hbuf, area.words);
}

typedef void (*fx_lstm_kernel_t)(const FxLstmArgs);
template <int L>
static fx_lstm_kernel_t pick_rows(int hpt, int tiles) {
  switch (hpt * 4 + tiles) {
    case 4 + 1: return fx_lstm_rows_kernel<L, 1, 1>;
    case 8 + 1: return fx_lstm_rows_kernel<L, 2, 1>;
    case 16 + 1: return fx_lstm_rows_kernel<L, 4, 1>;
    case 32 + 1: return fx_lstm_rows_kernel<L, 8, 1>;
    case 64 + 1: if constexpr (L <= 3) return fx_lstm_rows_kernel<L, 16, 1>; else return nullptr;
    case 64 + 2: if constexpr (L <= 3) return fx_lstm_rows_kernel<L, 16, 2>; else return nullptr;
    default: return nullptr;
  }
}
// one row, or rows one after the other: the sizes for which four units' weights and a tile of rows are far
// more than the registers hold (1024 units; four layers of 512: 725 us with spilled weights against 630
// for T = 32, B = 8).  Three layers of 512, T = 64, which spill less, row by row : one tile : two tiles, us:
//   B = 2 281 : 279 : 482, 4 551 : 321 : 518, 8 1 090 : 336 : 602, 9 1 260 : - : 740, 16 2 174 : - : 866
// two layers: B = 2 209 : 191 : 285, 8 804 : 228 : 346, 16 1 597 : - : 366.
template <int L>
static fx_lstm_kernel_t pick_serial(int hpt) {
  constexpr int U = FX_LSTM_UPW;
  switch (hpt) {
    case 1: return fx_lstm_stack_kernel<L, 1, U>;
    case 2: return fx_lstm_stack_kernel<L, 2, U>;
    case 4: return fx_lstm_stack_kernel<L, 4, U>;
    case 8: return fx_lstm_stack_kernel<L, 8, U>;
    case 16: return fx_lstm_stack_kernel<L, 16, U>;
    case 32: if constexpr (L <= 2) return fx_lstm_stack_kernel<L, 32, U>;
    default: return nullptr;
  }
}
typedef void (*fx_lstm_die_kernel_t)(const FxLstmArgs, int, int);
template <int L>
static fx_lstm_die_kernel_t pick_die(int hpt, int* threads) {
  switch (hpt) {
    case 2: *threads = FxLstmDie<1, L>::threads; return fx_lstm_die_kernel<1, L>;
    case 4: *threads = FxLstmDie<2, L>::threads; return fx_lstm_die_kernel<2, L>;
    case 8: *threads = FxLstmDie<4, L == 4 ? 2 : L>::threads; return fx_lstm_die_kernel<4, L == 4 ? 2 : L>;
    case 16: *threads = FxLstmDie<8, 1>::threads; return fx_lstm_die_kernel<8, 1>;
    default: return nullptr;
  }
}
enum LstmHandOver { LSTM_TAGS, LSTM_WORDS, LSTM_DIE };   // which area of the workspace
struct LstmLaunch { const void* kernel; int grid, threads, tiles; LstmHandOver over; int form; };   // tiles of rows a workgroup; 0: row by row
// the forms that serve these sizes, the fastest first
template <int L>
static int lstm_forms(const FxLstmArgs& a, LstmLaunch (&f)[5]) {
  const int hpt = a.H / 32;
  int n = 0, threads = 0;
  if (fx_lstm_die_fits(a.B, a.H, L))
    if (fx_lstm_die_kernel_t k = pick_die<L>(hpt, &threads)) {
      f[n++] = LstmLaunch{(const void*)k, FX_LSTM_DIES * FX_LSTM_DIE_WG, threads, 0, LSTM_DIE, FX_LSTM_FORM_DIE};
      f[n++] = LstmLaunch{(const void*)k, a.B * (L / fx_lstm_stage_layers(a.H, L)) * FX_LSTM_DIE_WG, threads, 0, LSTM_DIE, FX_LSTM_FORM_SPREAD};
    }
  if (a.B > 1)
    for (int tiles = 1; tiles <= 2; ++tiles) {
      const int groups = (a.B + 4 * tiles - 1) / (4 * tiles), cells = L * tiles < 4 ? L * tiles : 4;   // FxLstmRows
      if (fx_lstm_kernel_t k = pick_rows<L>(hpt, tiles)) f[n++] = LstmLaunch{(const void*)k, (a.H / 4) * groups, ((a.H >= 128 ? 8 : a.H / 16) + cells) * 64, tiles, LSTM_WORDS, tiles == 1 ? FX_LSTM_FORM_ROWS : FX_LSTM_FORM_ROWS2};
    }
  // two hidden units per workgroup: every workgroup fetches the step's vectors from the memory
  // side once, so fewer, larger workgroups fetch less, and sixteen gate sums fill the butterfly
  if (fx_lstm_kernel_t k = pick_serial<L>(hpt)) f[n++] = LstmLaunch{(const void*)k, a.H / FX_LSTM_UPW, FX_LSTM_BLOCK * FX_LSTM_UPW, 0, LSTM_TAGS, FX_LSTM_FORM_SINGLE};
  return n;
}

static thread_local int t_lstm_asked = FX_LSTM_FORM_ANY, t_lstm_taken = FX_LSTM_FORM_ANY;   // fx_set_lstm_form, fx_lstm_form
int fx_lstm_ask(int form) {
  const int before = t_lstm_asked;
  t_lstm_asked = form;
  return before;
}
int fx_lstm_taken() { return t_lstm_taken; }

static std::mutex g_lstm_mu;
static std::map<int, FxLstmGroups> g_lstm_groups;   // by device
static std::set<int> g_lstm_captured;               // devices on which a launch has been captured
// Workgroups of a form that a CU holds, and that it holds however their waves are dealt (fx_lstm_groups.h):
// facts of the code and the device, asked for once.
struct LstmFit { int per_cu, sure; };
static std::map<std::pair<int, const void*>, LstmFit> g_lstm_fit;
static hipError_t lstm_fit(int dev, const LstmLaunch& f, LstmFit* fit) {
  const void* k = f.kernel;
  auto it = g_lstm_fit.find({dev, k});
  if (it == g_lstm_fit.end()) {
    LstmFit v{};
    const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&v.per_cu, k, f.threads, 0);
    if (e != hipSuccess) return e;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&v.sure, k, (int)fx_lstm_block((uint32_t)f.threads), 0) != hipSuccess) {
      (void)hipGetLastError();
      v.sure = 1;
    }
    it = g_lstm_fit.emplace(std::make_pair(dev, k), v).first;
  }
  *fit = it->second;
  return hipSuccess;
}

// 0: launched; 1: shape outside what the kernel is built for; 2: the grid would not be resident
// all at once (every workgroup waits for values that all the others write); otherwise a HIP error code + 100.
int fx_launch_lstm_stack(const FxLstmArgs& args, int L, uint32_t* words_ctl, uint32_t* die_ctl, hipStream_t stream) {
  FxLstmArgs a = args;
  if (a.H < 32 || a.H % 32 != 0 || a.B < 1 || a.B > FX_LSTM_MAXB || L < 1 || L * a.B > FX_LSTM_BLOCK) return 1;
  LstmLaunch f[5];
  const int n = L == 1 ? lstm_forms<1>(a, f) : L == 2 ? lstm_forms<2>(a, f) : L == 3 ? lstm_forms<3>(a, f) : L == 4 ? lstm_forms<4>(a, f) : 0;
  if (n == 0) return 1;
  int dev = 0, cus = 0;
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  hipError_t e = hipGetDevice(&dev);
  if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  if (e != hipSuccess) return 100 + (int)e;
  if (hipStreamIsCapturing(stream, &cap) != hipSuccess) {
    (void)hipGetLastError();
    cap = hipStreamCaptureStatusNone;
  }
  const bool capturing = cap != hipStreamCaptureStatusNone;
  std::lock_guard<std::mutex> lock(g_lstm_mu);
  if (capturing) g_lstm_captured.insert(dev);
  // A captured launch is replayed whenever the program likes, beside any other: from the first one on,
  // every launch leaves half of the device free where a form of it can.
  const uint32_t device = (uint32_t)cus * FX_LSTM_CU / (g_lstm_captured.count(dev) ? 2u : 1u);
  const bool legacy = stream == nullptr || stream == hipStreamLegacy;
  const uint64_t id = legacy ? 0u : (uint64_t)(uintptr_t)stream;
  const uint64_t thread = stream == hipStreamPerThread ? (uint64_t)std::hash<std::thread::id>()(std::this_thread::get_id()) : 0u;
  FxLstmGroups& groups = g_lstm_groups[dev];
  const LstmLaunch* l = nullptr;
  uint32_t need = 0;
  const int asked = t_lstm_asked;
  for (int i = 0; i < n; ++i) {
    if (asked != FX_LSTM_FORM_ANY && asked != f[i].form) continue;
    // one tile of four rows a workgroup while that makes at most one workgroup for each CU, whose registers the
    // weights fill
    if (f[i].tiles == 1 && f[i].grid > cus && asked == FX_LSTM_FORM_ANY) continue;
    LstmFit fit;
    e = lstm_fit(dev, f[i], &fit);
    if (e != hipSuccess) return 100 + (int)e;
    if ((long)fit.per_cu * cus < f[i].grid) continue;
    const uint32_t want = fx_lstm_need((uint32_t)f[i].grid, (uint32_t)fit.sure);
    // A sequence on one die holds every die while its workgroups find their places: only where nothing else is about.
    // The same kernel spread over the chip holds what it uses and computes the same bits, so a size whose spread form needs
    // at most half of the device is computed by this kernel in every case: what a captured launch, or a call beside others,
    // computes is, to the bit, what a call by itself computes.
    const bool half = 2u * want <= (uint32_t)cus * FX_LSTM_CU;
    if (asked != FX_LSTM_FORM_ANY) {
      if (capturing && !half) continue;   // (a replay may run beside any other)
    } else if (f[i].over == LSTM_DIE) {
      if (a.T < fx_lstm_die_from(a.B, a.H, L)) continue;
      if (f[i].form == FX_LSTM_FORM_DIE ? capturing || want > device || a.T < fx_lstm_die_alone(a.B, a.H, L) || groups.others(id, thread) : !half) continue;
    }
    if (l && want >= need) continue;
    l = &f[i];
    need = want;
    if (need <= device) break;
  }
  if (!l) return asked == FX_LSTM_FORM_ANY ? 2 : 1;
  t_lstm_taken = l->form;
  uint32_t* areas[3] = {a.ctl, words_ctl, die_ctl ? die_ctl : a.ctl};
  std::swap(areas[0], areas[(int)l->over]);
  a.ctl = areas[0];
  a.ctl_other = areas[1];
  a.ctl_third = areas[2];
  a.hbuf = (uint64_t*)(a.ctl + FX_LSTM_CTL_WORDS);
  int spread = l->form == FX_LSTM_FORM_SPREAD ? 1 : 0;
  void* kargs[3] = {(void*)&a, (void*)&L, (void*)&spread};
  const dim3 grid((uint32_t)l->grid), block((uint32_t)l->threads);
  if (capturing) {
    e = hipLaunchKernel(l->kernel, grid, block, kargs, 0, stream);
    return e == hipSuccess ? 0 : 100 + (int)e;
  }
  auto record = [&](FxLstmGroups::Member& m) {
    if (!m.done) m.done = groups.event_to_use();
    if (!m.done) e = hipEventCreateWithFlags((hipEvent_t*)&m.done, hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventRecord((hipEvent_t)m.done, (hipStream_t)(uintptr_t)m.stream);
    return e == hipSuccess;
  };
  auto wait_for = [&](void* event) {
    e = hipStreamWaitEvent(stream, (hipEvent_t)event, 0);
    return e == hipSuccess;
  };
  bool joins = false;
  FxLstmGroups::Member& m = groups.admit(id, thread, need, device, legacy, &joins);
  m.last = ++groups.launches;
  if (joins && !(groups.close_late(record) && groups.wait(id, thread, wait_for))) {
    groups.withdraw();
    (void)hipGetLastError();
    return 100 + (int)e;
  }
  e = hipLaunchKernel(l->kernel, grid, block, kargs, 0, stream);
  // (a record costs launches in a row 1.3 - 2.5 us each; a completion event given to the kernel itself costs them
  // nothing, but some thousand such launches make every later call of the program, torch's as well, 5 us slower)
  if (e == hipSuccess && !m.late) (void)record(m);
  return e == hipSuccess ? 0 : 100 + (int)e;
}
