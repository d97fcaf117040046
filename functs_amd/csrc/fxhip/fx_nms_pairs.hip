// Class-aware NMS of boxes that are all candidates (mode 0 of fx_nms_desc: functs::nms and
// functs::batched_nms), as three small launches that use the whole chip where fx_sort_nms_kernel
// sorts, gathers, tests and walks in one workgroup per task (2 000 boxes, 260 kept: 140 us, of which
// 105 us are 400 000 overlap tests on one CU).  No launch waits for anything but the one before it.
//   1. fx_nms_rank_kernel    a workgroup per 16 boxes ranks them by counting the keys below theirs (the
//      keys of all rows in LDS, a sixty-fourth of them per quarter wave: n^2 comparisons over the chip
//      beat the log^2 n dependent stages of a sort in one workgroup up to the sizes that come here) and
//      writes their moved boxes, areas and indices to their places in score order;
//   2. fx_nms_pairs_kernel   a wave per 64 x 32 pairs: one word per box with its overlaps among 32 boxes
//      ahead of it in score order;
//   3. fx_nms_walk_kernel    a workgroup per task takes 64 boxes at a time in score order.  Which of a
//      chunk's boxes are overlapped by boxes kept before is, per earlier chunk, "word of the box and
//      kept boxes of that chunk": fifteen waves do that for the next chunk, as far as the kept boxes
//      are known, while the first wave adds the chunk just before its own and resolves it in rounds of
//      ballots.  The words come straight to registers, several chunks ahead.
// 2 000 boxes, 260 kept: rank 5.5, pairs 5.6, walk 21 us (0.5 us a chunk: barrier, the far boxes' bits out of
// LDS, two rounds, barrier), the call 157 -> 47 us.  Results are those of fx_sort_nms bit for bit: the same keys,
// the same overlap decisions, the same order of decisions.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../../include/fxhip.h"
#include "fx_nms.h"

#define FX_PAIRS_THREADS 1024u

namespace {

// Workspace of a task: [np] moved boxes, [np] areas, [np] rows, 64 words (the first: how many are
// candidates), [nw][np] 64-bit words of overlaps (of box j among the boxes of chunk c, c <= j / 64; the
// boxes of a chunk lie side by side); np = n rounded up to 64, nw = np / 64.
struct PairsWs {
  float4* box;
  float* area;
  uint32_t* row;
  uint32_t* count;
  uint64_t* over;
};
__host__ __device__ inline size_t pairs_ws_bytes(uint32_t n) {
  const size_t np = (n + 63u) & ~63u;
  return np * 24u + 256u + np * (np / 64u) * 8u;
}
__device__ __forceinline__ PairsWs pairs_ws(void* ws, uint32_t n, uint32_t task) {
  const uint32_t np = (n + 63u) & ~63u;
  uint8_t* p = (uint8_t*)ws + (size_t)task * pairs_ws_bytes(n);
  PairsWs w;
  w.box = (float4*)p;
  w.over = (uint64_t*)(p + (size_t)np * 16u);
  w.area = (float*)((uint8_t*)w.over + (size_t)np * (np / 64u) * 8u);
  w.row = (uint32_t*)(w.area + np);
  w.count = w.row + np;
  return w;
}

__global__ __launch_bounds__(FX_PAIRS_THREADS) void fx_nms_rank_kernel(const fx_nms_desc d) {
  extern __shared__ __attribute__((aligned(16))) uint64_t s_keys[];   // n, rounded up to 64
  __shared__ uint32_t s_rank[16];
  __shared__ uint32_t s_max, s_count;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const uint32_t n = d.rows, np = (n + 63u) & ~63u, nw = np >> 6;
  const uint32_t task = blockIdx.x / (4u * nw), blk = blockIdx.x - task * (4u * nw);
  const float* boxes = d.boxes + (int64_t)task * d.boxes_task_stride;
  const float* scores = d.scores + (int64_t)task * d.scores_task_stride;
  const int64_t* labels = d.labels ? d.labels + (int64_t)task * d.labels_task_stride : nullptr;
  const PairsWs ws = pairs_ws(d.workspace, n, task);
  if (tid < 16u) s_rank[tid] = 0u;
  if (tid == 0u) { s_max = 0u; s_count = 0u; }
  __syncthreads();
  // Every row's key, descending score and ascending row; a row that is no candidate sorts behind all
  // that are (the largest coordinate is taken over the candidates only).
  uint32_t my_max = 0u, my_count = 0u;
  for (uint32_t i = tid; i < np; i += FX_PAIRS_THREADS) {
    uint64_t key = ~0ull;
    if (i < n) {
      const float sc = scores[i];
      const float4 b = *(const float4*)(boxes + (size_t)i * 4u);
      const bool in = sc > d.score_thr;
      key = ((uint64_t)(in ? ~orderable(sc) : 0xffffffffu) << 32) | (uint64_t)i;
      if (in) {
        ++my_count;
        my_max = max(my_max, max(max(orderable(b.x), orderable(b.y)), max(orderable(b.z), orderable(b.w))));
      }
    }
    s_keys[i] = key;
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) my_max = max(my_max, (uint32_t)__shfl_xor((int)my_max, o, 64));
  my_count = fx_wave_sum(my_count, lane);
  if (lane == 0u) {
    atomicMax(&s_max, my_max);
    atomicAdd(&s_count, my_count);
  }
  __syncthreads();
  {
    // lane = candidate + 16 * quarter; the quarters of the waves take the keys one after the other, so that
    // the four that a wave reads at a time lie side by side
    const uint64_t mine = s_keys[(blk << 4) + (lane & 15u)];
    uint32_t below = 0u;
    const uint64_t* k = s_keys + wave * 4u + (lane >> 4);
#pragma unroll 4
    for (uint32_t i = 0; i < np; i += 64u) below += k[i] < mine ? 1u : 0u;
    below += fx_lane_xor<16u>(below, lane);
    below += fx_lane_xor<32u>(below, lane);
    if (lane < 16u) atomicAdd(&s_rank[lane], below);
  }
  __syncthreads();
  if (wave == 0u) {
    const uint32_t i = (blk << 4) + lane;
    if (lane < 16u && i < n) {
      const uint32_t r = s_rank[lane];
      const float class_step = from_orderable(s_max) + 1.0f;
      const float4 b = *(const float4*)(boxes + (size_t)i * 4u);
      const float off = (float)(labels ? (uint32_t)labels[i] : 0u) * class_step;
      const float4 m = make_float4(b.x + off, b.y + off, b.z + off, b.w + off);
      ws.box[r] = m;
      ws.area[r] = (m.z - m.x) * (m.w - m.y);
      ws.row[r] = i;
    }
    if (blk == 0u && lane == 0u) *ws.count = s_count;
  }
}

// grid: (columns of 32, four to a workgroup; chunks of 64 boxes; tasks)
__global__ __launch_bounds__(256) void fx_nms_pairs_kernel(const fx_nms_desc d) {
  __shared__ float4 s_box[4][32];
  __shared__ float s_area[4][32];
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const uint32_t n = d.rows, nw = (n + 63u) >> 6;
  const uint32_t chunk = blockIdx.y, col = blockIdx.x * 4u + wave;
  const PairsWs ws = pairs_ws(d.workspace, n, blockIdx.z);
  if (col > 2u * chunk + 1u) return;   // (waves share nothing)
  // every row has a box, those behind the candidates too: nothing waits for their number
  const uint32_t i = chunk * 64u + lane, j0 = col * 32u;
  if (lane < 32u) {
    const uint32_t j = min(j0 + lane, n - 1u);
    s_box[wave][lane] = ws.box[j];
    s_area[wave][lane] = ws.area[j];
  }
  const float4 q = ws.box[min(i, n - 1u)];
  const float area = ws.area[min(i, n - 1u)];
  const Box ib{q.x, q.y, q.z, q.w};
  // (no branch in the loop: the rare pairs that need the division are noted and decided behind it)
  uint32_t word = 0u, unsure = 0u;
#pragma unroll 8
  for (uint32_t j = 0; j < 32u; ++j) {
    const float4 p = s_box[wave][j];
    bool over, sure;
    overlaps_fast(ib, area, Box{p.x, p.y, p.z, p.w}, s_area[wave][j], d.iou_thr, over, sure);
    word |= over ? 1u << j : 0u;
    unsure |= sure ? 0u : 1u << j;
  }
  while (unsure != 0u) {
    const uint32_t j = (uint32_t)__builtin_ctz(unsure);
    const float4 p = s_box[wave][j];
    const bool over = overlaps(ib, area, Box{p.x, p.y, p.z, p.w}, s_area[wave][j], d.iou_thr);
    word = (word & ~(1u << j)) | (over ? 1u << j : 0u);
    unsure &= unsure - 1u;
  }
  ((uint32_t*)ws.over)[((size_t)(col >> 1) * (nw * 64u) + i) * 2u + (col & 1u)] = word;
}

#define FX_WALK_D 6u   // chunks that a wave's words are asked for ahead: they come from beyond the caches
template <uint32_t K> struct fx_slot { static constexpr uint32_t value = K; };
// W: words a wave holds per chunk, for 1 + 15 (W - 1) chunks or more.  The loads are unconditional (a place
// that has no word asks for one it does not use), so that how many are under way behind the one that is
// waited for is known when the kernel is compiled; and every step leaves the loop by itself.
template <uint32_t W>
__global__ __launch_bounds__(FX_PAIRS_THREADS) void fx_nms_walk_kernel(const fx_nms_desc d) {
  __shared__ uint32_t s_kept[FX_NMS_MAX_OUT];
  __shared__ uint64_t s_keep[64];      // boxes of a chunk that are kept
  __shared__ uint32_t s_dead[64][2];   // boxes of a chunk that a box kept two or more chunks before overlaps
  __shared__ uint32_t s_nk[2];         // boxes kept up to and with a chunk, by its parity: read behind the chunk's barrier
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = uni(tid >> 6);
  const uint32_t n = d.rows, nw = (n + 63u) >> 6, np = nw * 64u, task = blockIdx.x;
  const PairsWs ws = pairs_ws(d.workspace, n, task);
  const uint32_t count = uni(*ws.count), chunks = (count + 63u) >> 6;
  if (tid < 64u) {
    s_dead[tid][0] = 0u;
    s_dead[tid][1] = 0u;
  }
  uint64_t held[FX_WALK_D][W];
  // First wave: words of chunk c in itself and in the chunk before.  Wave v: words of chunk c + 1 in
  // chunks v - 1, v + 14, ...  (Relaxed atomic loads: plain ones are moved down to where they are used.)
  auto ask = [&](uint32_t c, uint64_t (&to)[W]) __attribute__((always_inline)) {
    const uint32_t chunk = wave == 0u ? c : c + 1u;
#pragma unroll
    for (uint32_t k = 0; k < W; ++k) {
      const uint32_t w = wave == 0u ? (k == 0u ? c : c - 1u) : wave - 1u + 15u * k;
      const bool want = chunk < chunks && (wave == 0u ? k < 2u && w <= c : w < c);
      // (the place of a word that is not wanted is one line that stays in the cache: a single CU gets
      // the words at some 50 GB/s, which bounds the walk)
      const uint64_t* at = ws.over + uni(want ? w * np + chunk * 64u : 0u);
      to[k] = __hip_atomic_load(at + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    }
  };
  ask(0u, held[0]); ask(1u, held[1]); ask(2u, held[2]); ask(3u, held[3]); ask(4u, held[4]); ask(5u, held[5]);
  __syncthreads();
  uint32_t nk = 0u;
  uint64_t before = 0ull;   // first wave: kept boxes of the chunk before
  if (wave == 0u) __builtin_amdgcn_s_setprio(3);   // the others only have to be done before the next chunk
  // walks chunk c, whose words are in slot k; true: it was the last one
  auto step = [&](auto slot, uint32_t c) __attribute__((always_inline)) -> bool {
    constexpr uint32_t k = decltype(slot)::value;
    if (wave == 0u) {
      const uint32_t m = min(64u, count - c * 64u);
      const uint64_t in = held[k][0] & ((1ull << lane) - 1ull);   // overlapping boxes of the chunk ahead of this one
      const uint64_t valid = m >= 64u ? ~0ull : (1ull << m) - 1ull;
      const uint64_t far = ((uint64_t)uni(s_dead[c][1]) << 32) | (uint64_t)uni(s_dead[c][0]);
      const uint64_t near = __ballot((held[k][1] & before) != 0ull);
      // All boxes decide together: one whose overlapping predecessors are all dead is kept, the ones it
      // overlaps are dead; the first undecided box always decides, and one or two rounds settle a chunk.
      uint64_t keptm = 0ull, open = valid & ~(far | near);
      while (open != 0ull) {
        const bool mine = ((open >> lane) & 1ull) != 0ull;
        const uint64_t kept = __ballot(mine && (in & open) == 0ull);
        const uint64_t dead = __ballot(mine && (in & kept) != 0ull);
        keptm |= kept;
        open &= ~(kept | dead);
      }
      const uint32_t rank = (uint32_t)__popcll(keptm & ((1ull << lane) - 1ull));
      const bool keep = ((keptm >> lane) & 1ull) != 0ull && rank < d.max_num - nk;
      if (keep) s_kept[nk + rank] = c * 64u + lane;
      before = __ballot(keep);
      nk += (uint32_t)__popcll(before);
      if (lane == 0u) {
        s_keep[c] = before;
        s_nk[k & 1u] = nk;
      }
    } else if (c + 1u < chunks) {
      uint64_t kept[W];
#pragma unroll
      for (uint32_t q = 0; q < W; ++q) kept[q] = s_keep[min(wave - 1u + 15u * q, 63u)];   // (all reads in flight together)
      uint64_t over = 0ull;
#pragma unroll
      for (uint32_t q = 0; q < W; ++q) over |= wave - 1u + 15u * q < c ? held[k][q] & kept[q] : 0ull;
      const bool dead = over != 0ull;
      const uint64_t x = __ballot(dead);
      if (lane < 2u && x != 0ull) atomicOr(&s_dead[c + 1u][lane], (uint32_t)(x >> (32u * lane)));
    }
    ask(c + FX_WALK_D, held[k]);
    __syncthreads();
    if (wave != 0u) nk = uni(s_nk[k & 1u]);
    return nk >= d.max_num || c + 1u >= chunks;
  };
  static_assert(FX_WALK_D == 6u, "one call per slot (an index that the compiler does not know would put the words into scratch memory)");
  for (uint32_t c = 0; chunks > 0u; c += FX_WALK_D) {
    if (step(fx_slot<0>(), c)) break;
    if (step(fx_slot<1>(), c + 1u)) break;
    if (step(fx_slot<2>(), c + 2u)) break;
    if (step(fx_slot<3>(), c + 3u)) break;
    if (step(fx_slot<4>(), c + 4u)) break;
    if (step(fx_slot<5>(), c + 5u)) break;
  }
  // (system scope: a count in pinned host memory goes through to the host, which may be polling it)
  if (tid == 0u) __hip_atomic_store(d.n_out + task, nk, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  const float* boxes = d.boxes + (int64_t)task * d.boxes_task_stride;
  const float* scores = d.scores + (int64_t)task * d.scores_task_stride;
  const int64_t* labels = d.labels ? d.labels + (int64_t)task * d.labels_task_stride : nullptr;
  float* dets = d.dets + (size_t)task * d.max_num * 5u;
  int64_t* out_labels = d.out_labels + (size_t)task * d.max_num;
  int64_t* out_index = d.out_index ? d.out_index + (size_t)task * d.max_num : nullptr;
  for (uint32_t k = tid; k < d.max_num; k += FX_PAIRS_THREADS) {   // rows past the kept ones are zero: the outputs have a fixed shape
    const bool live = k < nk;
    const uint32_t i = live ? ws.row[s_kept[live ? k : 0u]] : 0u;
    const float4 b = live ? *(const float4*)(boxes + (size_t)i * 4u) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    float* o = dets + (size_t)k * 5u;
    o[0] = b.x; o[1] = b.y; o[2] = b.z; o[3] = b.w;
    o[4] = live ? scores[i] : 0.0f;
    out_labels[k] = live && labels ? (int64_t)(uint32_t)labels[i] : 0;
    if (out_index) out_index[k] = live ? (int64_t)i : 0;
  }
}

}  // namespace

size_t fx_nms_pairs_ws_bytes(int n_tasks, uint32_t rows) { return (size_t)n_tasks * pairs_ws_bytes(rows); }

// d: mode 0 without counts, 1 .. FX_NMS_PAIRS_MAX_ROWS rows; 0: launched; otherwise a HIP error code + 100
int fx_launch_nms_pairs(const fx_nms_desc& d, hipStream_t stream) {
  const uint32_t nw = (d.rows + 63u) / 64u;
  hipLaunchKernelGGL(fx_nms_rank_kernel, dim3((uint32_t)d.n_tasks * 4u * nw), dim3(FX_PAIRS_THREADS), (size_t)nw * 64u * 8u, stream, d);
  hipLaunchKernelGGL(fx_nms_pairs_kernel, dim3((2u * nw + 3u) / 4u, nw, (uint32_t)d.n_tasks), dim3(256), 0, stream, d);
  auto* walk = nw <= 31u ? fx_nms_walk_kernel<2> : nw <= 46u ? fx_nms_walk_kernel<3> : fx_nms_walk_kernel<5>;
  hipLaunchKernelGGL(walk, dim3((uint32_t)d.n_tasks), dim3(FX_PAIRS_THREADS), 0, stream, d);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : 100 + (int)e;
}
