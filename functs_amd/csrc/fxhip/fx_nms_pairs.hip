// Class-aware NMS of boxes that are all candidates (mode 0 of fx_nms_desc: functs::nms and
// functs::batched_nms), as three small launches that use the whole chip where fx_sort_nms_kernel
// sorts, gathers, tests and walks in one workgroup per task (2 000 boxes apart from each other: 82 us, most of
// it 1 700 000 overlap tests on one CU).  No launch waits for anything but the one before it.
//   1. fx_nms_rank_kernel    a workgroup per 16 boxes ranks them by counting the keys below theirs (the
//      keys of all rows in LDS, a sixty-fourth of them per quarter wave: n^2 comparisons over the chip
//      beat the log^2 n dependent stages of a sort in one workgroup up to the sizes that come here) and
//      writes their moved boxes, areas and indices to their places in score order;
//   2. fx_nms_pairs_kernel   a wave per 64 x 32 pairs: one word per box with its overlaps among 32 boxes
//      ahead of it in score order;
//   3. up to 16 chunks of 64 boxes, and where few are to be kept, fx_nms_walk_kernel: a workgroup per task
//      takes a chunk at a time in score order.  Which of a chunk's boxes are overlapped by boxes kept before is, per earlier chunk,
//      "word of the box and kept boxes of that chunk": fifteen waves do that for the next chunk, as far as
//      the kept boxes are known, while the first wave adds the chunk just before its own and resolves it in
//      rounds of ballots.  The words come straight to registers, several chunks ahead.
//      Otherwise fx_nms_resolve_kernel, a workgroup per chunk.  A box is dead when a kept box ahead of it
//      overlaps it, and kept when every overlapping box ahead of it is dead; chunks publish what they have
//      decided as soon as they have, and look at what the chunks ahead have published, so the chunks are
//      resolved side by side: the wait is for as many exchanges as a chain of overlaps has links, at most
//      one a chunk, not for every chunk in turn.
// Microseconds of the three launches back to back, walk : resolve, one image (2 000 boxes: rank 5.6, pairs 5.4, walk
// 21 or resolve 10): 2 000 proposals of 60 objects 31.6 : 27.1, dense crowd 26.4 : 23.8, apart from each other
// 24.2 : 17.3, each overlapping the next 23.3 : 17.1; 4 096: 73 : 44, 40 : 38, 37 : 30, 36 : 30; 8 images of 2 000:
// 53 : 51, 47 : 47, 45 : 39, 44 : 39.  What is left of resolve is its exchanges, some 1.1 us each: a store's way to
// the other dies, half a look, the words through LDS.  At 1 000 boxes the two are level (19.6 : 19.7), at 500 the
// walk is faster (15.1 : 16.3); where max_num is reached early the walk ends early (crowd of 2 000, 300 kept of the
// first 450: 17.1 : 19.0), hence the rule on max_num.  Call of 2 000 boxes, 260 kept: 46.5 -> 37.5 us.
// Results are those of fx_sort_nms bit for bit: the same keys, the same overlap decisions, and the one result
// that decisions in score order have.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../../include/fxhip.h"
#include "fx_nms.h"

#define FX_PAIRS_THREADS 1024u

namespace {

// Workspace of a task: [np] moved boxes, [np] areas, [np] rows, 64 words (the first: how many are
// candidates), [nw][np] 64-bit words of overlaps (of box j among the boxes of chunk c, c <= j / 64; the
// boxes of a chunk lie side by side), [64] pairs of 64-bit words (the boxes of a chunk that are kept, those that
// are dead, as far as they are decided); np = n rounded up to 64, nw = np / 64.
struct PairsWs {
  float4* box;
  float* area;
  uint32_t* row;
  uint32_t* count;
  uint64_t* over;
  uint64_t* state;
};
__host__ __device__ inline size_t pairs_ws_bytes(uint32_t n) {
  const size_t np = (n + 63u) & ~63u;
  return np * 24u + 256u + 1024u + np * (np / 64u) * 8u;
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
  w.state = (uint64_t*)(w.count + 64u);
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
// RESOLVE: fx_nms_resolve_kernel follows, whose workgroups find the results cleared (the walk's one workgroup fills them to
// the end itself: of few boxes this launch has few threads for it.  200 boxes, three launches: 12.8 us so, 13.0 cleared here,
// the call 29.0 against 29.5 to 31)
template <bool RESOLVE>
__global__ __launch_bounds__(256) void fx_nms_pairs_kernel(const fx_nms_desc d) {
  __shared__ float4 s_box[4][32];
  __shared__ float s_area[4][32];
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const uint32_t n = d.rows, nw = (n + 63u) >> 6;
  const uint32_t chunk = blockIdx.y, col = blockIdx.x * 4u + wave;
  const PairsWs ws = pairs_ws(d.workspace, n, blockIdx.z);
  if constexpr (RESOLVE) {
    // the results start out as zeros (rows past the kept ones stay so: the outputs have a fixed shape), the
    // chunks as undecided; the next launch is the first to touch either
    const uint32_t at = (chunk * gridDim.x + blockIdx.x) * 256u + threadIdx.x, step = gridDim.x * gridDim.y * 256u;
    float* dets = d.dets + (size_t)blockIdx.z * d.max_num * 5u;
    int64_t* out_labels = d.out_labels + (size_t)blockIdx.z * d.max_num;
    int64_t* out_index = d.out_index ? d.out_index + (size_t)blockIdx.z * d.max_num : nullptr;
    for (uint32_t k = at; k < d.max_num * 5u; k += step) dets[k] = 0.0f;
    for (uint32_t k = at; k < d.max_num; k += step) {
      out_labels[k] = 0;
      if (out_index) out_index[k] = 0;
    }
    if (at < 128u) ws.state[at] = 0ull;
  }
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

__device__ __forceinline__ uint64_t uni64(uint64_t v) { return ((uint64_t)uni((uint32_t)(v >> 32)) << 32) | (uint64_t)uni((uint32_t)v); }

// The boxes of a chunk that can be decided, round after round: one with a kept overlapping predecessor (`in`:
// those in the chunk) is dead, one whose overlapping predecessors are all dead and that waits for none outside
// the chunk is kept.
__device__ __forceinline__ void resolve_chunk(uint64_t in, uint64_t waits, uint32_t lane, uint64_t& kept, uint64_t& dead) {
  for (;;) {
    const bool open = (((kept | dead) >> lane) & 1ull) == 0ull;
    const bool is_dead = open && (in & kept) != 0ull;
    const bool is_kept = open && !is_dead && ((waits >> lane) & 1ull) == 0ull && (in & ~dead) == 0ull;
    const uint64_t nd = __ballot(is_dead), nk = __ballot(is_kept);
    if ((nd | nk) == 0ull) return;
    dead |= nd;
    kept |= nk;
  }
}

// Wave 0 decides the chunk's boxes; waves 1 .. 15 hold the words of the chunk's boxes among the chunks ahead,
// W each, look at the state of those and tell wave 0 which boxes are dead for it (s_dead) and which still wait
// (s_wait).  A wave writes the former before the latter and wave 0 reads them the other way round: LDS serves a
// wave's accesses in order, so a box that waits no more is known to be dead if it is.
// A workgroup waits for workgroups of lower number only.  All waits are bounded: one that is given up after
// spin_limit looks makes wave 0 resolve the chunks from the first on by itself, from the words alone.
// max_num boxes kept ahead of a chunk end it: none of its boxes would be among the results, whatever it is that the
// boxes of the chunks ahead still wait for.
#define FX_GAVE_UP 1u
#define FX_FULL 2u
template <uint32_t W>
__global__ __launch_bounds__(FX_PAIRS_THREADS) void fx_nms_resolve_kernel(const fx_nms_desc d, const uint32_t spin_limit) {
  __shared__ uint64_t s_keep[64];   // kept boxes of the chunks up to this one
  __shared__ uint64_t s_wait[16];
  __shared__ uint32_t s_dead[2];
  __shared__ uint32_t s_ahead[16];   // boxes that a wave has seen kept
  __shared__ uint32_t s_stop;        // FX_GAVE_UP, FX_FULL
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = uni(tid >> 6);
  const uint32_t n = d.rows, nw = (n + 63u) >> 6, np = nw * 64u, task = blockIdx.x / nw, c = blockIdx.x - task * nw;
  const PairsWs ws = pairs_ws(d.workspace, n, task);
  // asked for together: how many are candidates, the words (written for every row), the rows of this chunk
  const uint32_t mine = c * 64u + (tid >> 4), part = tid & 15u;
  const uint32_t n_cand = *ws.count, row = ws.row[min(mine, n - 1u)];
  uint64_t word[W];
#pragma unroll
  for (uint32_t k = 0; k < W; ++k) {
    const uint32_t l = wave == 0u ? c : wave - 1u + 15u * k;
    word[k] = (wave == 0u ? k == 0u : l < c) ? ws.over[(size_t)l * np + c * 64u + lane] : 0ull;
  }
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  const uint32_t count = uni(n_cand), chunks = (count + 63u) >> 6;
  if (c >= chunks) {
    // (system scope: a count in pinned host memory goes through to the host, which may be polling it)
    if (count == 0u && c == 0u && tid == 0u) __hip_atomic_store(d.n_out + task, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    return;
  }
  // what the rows of this chunk will hold, sixteen threads a box, asked for ahead of the wait
  uint32_t label = 0u;
  float value = 0.0f;
  if (mine < count) {
    if (part < 4u) value = d.boxes[(int64_t)task * d.boxes_task_stride + (size_t)row * 4u + part];
    if (part == 4u) value = d.scores[(int64_t)task * d.scores_task_stride + row];
    if (part == 5u && d.labels) label = (uint32_t)d.labels[(int64_t)task * d.labels_task_stride + row];
  }
  if (tid < 16u) s_wait[tid] = tid != 0u && tid - 1u < c ? ~0ull : 0ull;
  if (tid < 2u) s_dead[tid] = 0u;
  if (tid < 16u) s_ahead[tid] = 0u;
  if (tid == 0u) s_stop = 0u;
  __syncthreads();
  uint64_t* state = ws.state;
  if (wave == 0u) {
    __builtin_amdgcn_s_setprio(3);   // what this wave decides is what others wait for
    const uint64_t in = word[0] & ((1ull << lane) - 1ull);
    const uint32_t m = min(64u, count - c * 64u);
    uint64_t kept = 0ull, dead = m >= 64u ? 0ull : ~((1ull << m) - 1ull);
    for (;;) {
      uint64_t w = __hip_atomic_load(&s_wait[lane & 15u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      const uint32_t d0 = __hip_atomic_load(&s_dead[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      const uint32_t d1 = __hip_atomic_load(&s_dead[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      uint32_t ahead = __hip_atomic_load(&s_ahead[lane & 15u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      if (uni(__hip_atomic_load(&s_stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) != 0u) break;
      ahead += fx_lane_xor<1u>(ahead, lane);
      ahead += fx_lane_xor<2u>(ahead, lane);
      ahead += fx_lane_xor<4u>(ahead, lane);
      ahead += fx_lane_xor<8u>(ahead, lane);
      if (uni(ahead) >= d.max_num) {
        if (lane == 0u) __hip_atomic_store(&s_stop, FX_FULL, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        break;
      }
      uint32_t w0 = (uint32_t)w, w1 = (uint32_t)(w >> 32);
      w0 |= fx_lane_xor<1u>(w0, lane); w1 |= fx_lane_xor<1u>(w1, lane);
      w0 |= fx_lane_xor<2u>(w0, lane); w1 |= fx_lane_xor<2u>(w1, lane);
      w0 |= fx_lane_xor<4u>(w0, lane); w1 |= fx_lane_xor<4u>(w1, lane);
      w0 |= fx_lane_xor<8u>(w0, lane); w1 |= fx_lane_xor<8u>(w1, lane);
      const uint64_t waits = ((uint64_t)uni(w1) << 32) | (uint64_t)uni(w0), was = kept | dead;
      dead |= (((uint64_t)uni(d1) << 32) | (uint64_t)uni(d0)) & ~kept;
      resolve_chunk(in, waits, lane, kept, dead);
      if ((kept | dead) != was && lane < 2u)
        __hip_atomic_store(state + 2u * c + lane, lane == 0u ? kept : dead, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (~(kept | dead) == 0ull) break;
    }
    if (lane == 0u) s_keep[c] = kept;
  } else {
    uint32_t open = 0u;   // chunks of this wave that are not decided to the last box
#pragma unroll
    for (uint32_t k = 0; k < W; ++k) open |= wave - 1u + 15u * k < c ? 1u << k : 0u;
    uint64_t waited = ~0ull;
    uint32_t closed_kept = 0u, counted = 0u;
    bool dead = false;
    for (uint32_t polls = 0; open != 0u; ++polls) {
      if (uni(__hip_atomic_load(&s_stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) != 0u) break;
      if (polls >= spin_limit) {
        if (lane == 0u) __hip_atomic_store(&s_stop, FX_GAVE_UP, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        break;
      }
      uint64_t kept[W], gone[W];
#pragma unroll
      for (uint32_t k = 0; k < W; ++k) {
        const uint64_t* at = state + 2u * ((open >> k) & 1u ? wave - 1u + 15u * k : 0u);
        kept[k] = __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        gone[k] = __hip_atomic_load(at + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      bool waits = false;
      uint32_t seen = closed_kept;
#pragma unroll
      for (uint32_t k = 0; k < W; ++k) {
        if (((open >> k) & 1u) == 0u) continue;
        // (what one lane has seen: were some to see an earlier state than the one that closes the chunk, they would not look again)
        kept[k] = uni64(kept[k]);
        gone[k] = uni64(gone[k]);
        dead = dead || (word[k] & kept[k]) != 0ull;
        waits = waits || (word[k] & ~(kept[k] | gone[k])) != 0ull;
        seen += (uint32_t)__popcll(kept[k]);
        if (~(kept[k] | gone[k]) == 0ull) {
          open &= ~(1u << k);
          closed_kept += (uint32_t)__popcll(kept[k]);
          if (lane == 0u) s_keep[wave - 1u + 15u * k] = kept[k];
        }
      }
      if (seen != counted) {
        counted = seen;
        if (lane == 0u) __hip_atomic_store(&s_ahead[wave], seen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
      const uint64_t now = __ballot(waits && !dead);
      if (now != waited) {
        waited = now;
        const uint64_t x = __ballot(dead);
        if (lane < 2u) __hip_atomic_fetch_or(&s_dead[lane], (uint32_t)(x >> (32u * lane)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        if (lane == 0u) __hip_atomic_store(&s_wait[wave], now, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
    }
  }
  __syncthreads();
  const uint32_t stop = uni(s_stop);
  if (stop == FX_FULL) {
    // (the other boxes of this chunk are no results either way: nobody is to wait for them)
    if (tid == 0u) __hip_atomic_store(state + 2u * c + 1u, ~0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (c + 1u == chunks && tid == 0u) __hip_atomic_store(d.n_out + task, d.max_num, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    return;
  }
  if (stop == FX_GAVE_UP) {
    if (wave == 0u) {
      for (uint32_t e = 0; e <= c; ++e) {
        uint64_t over = 0ull;
        for (uint32_t l = 0; l < e; ++l) over |= ws.over[(size_t)l * np + e * 64u + lane] & s_keep[l];
        const uint32_t m = min(64u, count - e * 64u);
        uint64_t kept = 0ull, dead = __ballot(over != 0ull) | (m >= 64u ? 0ull : ~((1ull << m) - 1ull));
        resolve_chunk(ws.over[(size_t)e * np + e * 64u + lane] & ((1ull << lane) - 1ull), 0ull, lane, kept, dead);
        if (lane == 0u) s_keep[e] = kept;
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        if (e == c && lane < 2u)
          __hip_atomic_store(state + 2u * c + lane, lane == 0u ? kept : ~kept, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    __syncthreads();
  }
  const uint64_t keep = uni64(s_keep[c]);
  const uint32_t ahead = uni(fx_wave_sum(lane < c ? (uint32_t)__popcll(s_keep[lane]) : 0u, lane));
  if (c + 1u == chunks && tid == 0u)
    __hip_atomic_store(d.n_out + task, min(ahead + (uint32_t)__popcll(keep), d.max_num), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  const uint32_t box = tid >> 4, at = ahead + (uint32_t)__popcll(keep & ((1ull << box) - 1ull));
  if (((keep >> box) & 1ull) == 0ull || at >= d.max_num) return;
  if (part < 5u) d.dets[((size_t)task * d.max_num + at) * 5u + part] = value;
  if (part == 5u) d.out_labels[(size_t)task * d.max_num + at] = (int64_t)label;
  if (part == 6u && d.out_index) d.out_index[(size_t)task * d.max_num + at] = (int64_t)row;
}

}  // namespace

size_t fx_nms_pairs_ws_bytes(int n_tasks, uint32_t rows) { return (size_t)n_tasks * pairs_ws_bytes(rows); }

// d: mode 0 without counts, 1 .. FX_NMS_PAIRS_MAX_ROWS rows; 0: launched; otherwise a HIP error code + 100
int fx_launch_nms_pairs(const fx_nms_desc& d, uint32_t spin_limit, hipStream_t stream) {
  const uint32_t nw = (d.rows + 63u) / 64u;
  hipLaunchKernelGGL(fx_nms_rank_kernel, dim3((uint32_t)d.n_tasks * 4u * nw), dim3(FX_PAIRS_THREADS), (size_t)nw * 64u * 8u, stream, d);
  // level at 16 chunks, and ahead of each other on either side of it; with few to be kept the walk may end early (top)
  const bool by_chunks = nw > 16u && (uint64_t)d.max_num * 4u >= d.rows;
  auto* pairs = by_chunks ? fx_nms_pairs_kernel<true> : fx_nms_pairs_kernel<false>;
  hipLaunchKernelGGL(pairs, dim3((2u * nw + 3u) / 4u, nw, (uint32_t)d.n_tasks), dim3(256), 0, stream, d);
  if (by_chunks) {
    auto* resolve = nw <= 31u ? fx_nms_resolve_kernel<2> : nw <= 46u ? fx_nms_resolve_kernel<3> : fx_nms_resolve_kernel<5>;
    hipLaunchKernelGGL(resolve, dim3((uint32_t)d.n_tasks * nw), dim3(FX_PAIRS_THREADS), 0, stream, d, spin_limit);
  } else {
    auto* walk = nw <= 31u ? fx_nms_walk_kernel<2> : nw <= 46u ? fx_nms_walk_kernel<3> : fx_nms_walk_kernel<5>;
    hipLaunchKernelGGL(walk, dim3((uint32_t)d.n_tasks), dim3(FX_PAIRS_THREADS), 0, stream, d);
  }
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : 100 + (int)e;
}
