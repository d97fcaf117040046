// Detection tail in ONE launch for all tasks (images): candidate selection by score threshold,
// sort by descending score, class-aware greedy NMS, top-k.  What the reference runs after its row
// compaction as a chain of ATen / torchvision kernels with host synchronisations in between
// (nonzero, index, max, sort, torchvision::nms, slicing: functs/benchmark/ai_model/yolov3/
// yolov3_bbox.py:104-179, functs/benchmark/ai_model/ssd/ssd_bbox.py:163-214).
//
// `slices` workgroups of 1024 threads per task share the scan of its scores; the last of them to
// finish (a ticket counter: nobody waits for anybody) does the rest alone, in LDS:
//   1. candidates whose score passes the threshold become 64-bit keys (inverted orderable score
//      bits : candidate index), collected in LDS by each workgroup and appended to the task's
//      key buffer in the workspace - their order of arrival does not matter, the index in the
//      key restores it;
//   2. keys in ascending order: descending score, equal scores by ascending index (a stable descending sort): by
//      buckets of the score for up to FX_NMS_FEW candidates, whose boxes come with their keys, else a bitonic sort;
//   3. candidates are taken 64 at a time in that order.  Each is tested against the kept list
//      (16 waves, every 16th kept box each), the overlaps inside the chunk become one 64-bit word
//      per candidate (its overlapping predecessors), and one wave resolves the chunk: all
//      candidates decide together in rounds, as many as the longest chain of overlaps.  The
//      walk ends when max_num boxes are kept: later candidates cannot change earlier decisions.
// What is left behind the scan runs on one CU an image and is bound by what that CU issues and by the trips between its
// steps.  16 images of 8 500 rows, 80 classes, about 760 candidates each: 23.8 us; 27.9 with the sort for all, factors and
// boxes gathered by the last workgroup, the rows written in the walk (whose barriers then wait for the stores) and
// the walk's overlaps by the division.  128 boxes of one image, one workgroup, nothing handed over: 12.1 us, 13.1.
// Few candidates that several workgroups find pay for the buckets and the hand-over: calls of one image of 8 500 rows with 8 / 100 /
// 200 / 700 candidates 14.3 / 16.7 / 16.8 / 17.6 us, with the sort and the last workgroup's gather 13.0 / 15.8 / 17.3 / 21.2.  (Up to 128
// candidates ordered by counting, eight threads each, 13.8 / 16.5, was 0.2 to 0.4 slower at 200 to 300: the kernel grows.)
// The workspace counters are zero when a launch starts and zero again when it ends.
// The number of valid rows per task is read from memory (device or pinned host), so the count a
// preceding compaction produced never has to reach the host.
// Arithmetic of an overlap test, in float32 and in this order (no contraction):
//   box + label * (max coordinate + 1);  area = (x2 - x1) * (y2 - y1);
//   inter = max(0, min(x2) - max(x1)) * max(0, min(y2) - max(y1));  iou = inter / ((area_i + area_j) - inter) > thr
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <limits>
#include <mutex>
#include <type_traits>

#include "../../../include/fxhip.h"
#include "fx_nms.h"

// a hook for timing the phases of a task's last workgroup from a test program; nothing in the library
#ifndef FX_NMS_STAMP
#define FX_NMS_STAMP(k)
#endif

#define FX_NMS_THREADS 1024u
#define FX_NMS_CHUNK 64u
#define FX_NMS_OWN 2u           // candidates a thread of the finishing workgroup holds where it orders by buckets
#define FX_NMS_FEW (FX_NMS_OWN * FX_NMS_THREADS)
#define FX_NMS_BUCKET_BITS 11u
#define FX_NMS_BUCKETS (1u << FX_NMS_BUCKET_BITS)
#define FX_NMS_CROWD 48u        // candidates in a bucket that compare themselves with each other
// key capacity from which LDS holds what a walk of FX_NMS_FEW candidates needs
#define FX_NMS_ROOMY 16384u
static_assert(FX_NMS_ROOMY * 8u >= FX_NMS_BUCKETS * 4u + FX_NMS_FEW * 56u, "the finishing workgroup's arrays lie in the keys' memory");

namespace {

// one stage of the bitonic network on a key a lane, partners J lanes apart: the lower lane keeps
// the smaller key where the run ascends
template <uint32_t J>
__device__ __forceinline__ uint64_t bitonic_step(uint64_t key, bool up, uint32_t lane) {
  const uint64_t other = ((uint64_t)fx_lane_xor<J>((uint32_t)(key >> 32), lane) << 32) | (uint64_t)fx_lane_xor<J>((uint32_t)key, lane);
  const bool keep_min = ((lane & J) == 0u) == up;
  return ((key < other) == keep_min) ? key : other;
}

// workspace: per task FX_NMS_WS_WORDS counters (candidates, finished slices, largest coordinate,
// row count + 1; zero between launches) in front of all tasks' key buffers, behind which lie FX_NMS_FEW boxes a task
// (of the first candidates, in the keys' order of arrival)
#define FX_NMS_WS_WORDS 64u

// ---- a detection head's maps as the source of the rows ----
// Rows lie level after level, in a level cell after cell, in a cell anchor after anchor, as the head's permutation
// puts them (yolov3_bbox.py:211-220).  Class scores of one (level, anchor) are C * cells consecutive elements of an
// image's map; a wave reads them in groups of 256 that never span two of these runs, so what a wave needs to know
// about its group is uniform.
// Four 608 x 608 images, 80 classes, about 700 candidates each, cold lines: 21.7 us, of which the scan's 28 MB are 6.7 behind
// 2 of start; the functors and the tail this stands for (rows across their order 38.5, row stream 16.8, tail 26.1) 81.4,
// and the call 97 -> 35 us.  One image 19.8 (128 workgroups scan it; 64: 20.5, 256: 21.7, they queue up for the ticket).
struct HeadLevel {
  const float *map, *base, *shift;
  uint32_t cells, anchors, row0;     // row0: rows of the levels before it
  uint32_t group0, run_groups;       // groups of the levels before it; groups of a run
  uint32_t cells_magic, cells_shift, anchors_magic, anchors_shift, run_magic, run_shift;
};
struct HeadMaps {
  HeadLevel lv[FX_HEAD_LEVELS];
  uint32_t n_levels, groups, width;  // groups of an image; attributes of a row (5 + classes)
  uint32_t c_magic, c_shift;         // division by the number of classes
  float keep_thr, logit_lo;          // no element below logit_lo passes the score threshold
  const float* strides;
};
struct NoMaps {};
__device__ __forceinline__ uint32_t divisor_magic(const HeadMaps& h) { return h.c_magic; }
__device__ __forceinline__ uint32_t divisor_shift(const HeadMaps& h) { return h.c_shift; }
__device__ __forceinline__ uint32_t divisor_magic(const NoMaps&) { return 0u; }
__device__ __forceinline__ uint32_t divisor_shift(const NoMaps&) { return 0u; }

// A class score's place, from its number (256 x the groups in front of its run, and its number in the run): level by selects
// (lanes differ), then the row's planes and tables.
struct HeadRow {
  const float* at;      // attribute 0; attribute k lies k * cells behind it
  uint32_t cells, row, label;
  const float *base, *shift, *stride;
};
__device__ __forceinline__ HeadRow head_row(const HeadMaps& h, uint32_t task, uint32_t number) {
  HeadLevel v = h.lv[0];
#pragma unroll
  for (uint32_t l = 1; l < FX_HEAD_LEVELS; ++l)
    if (l < h.n_levels && (number >> 8) >= h.lv[l].group0) v = h.lv[l];
  const uint32_t a = fx_fastdiv((number >> 8) - v.group0, v.run_magic, v.run_shift), in_run = number - (v.group0 + a * v.run_groups) * 256u;
  const uint32_t label = fx_fastdiv(in_run, v.cells_magic, v.cells_shift), cell = in_run - label * v.cells, row = v.row0 + cell * v.anchors + a;
  return HeadRow{v.map + (size_t)(task * v.anchors + a) * h.width * v.cells + cell, v.cells, row, label, v.base + a * 4u,
                 v.shift + (size_t)cell * 4u, h.strides + row};
}
// the number of (row, label), as above
__device__ __forceinline__ uint32_t head_number(const HeadMaps& h, uint32_t row, uint32_t label) {
  HeadLevel v = h.lv[0];
#pragma unroll
  for (uint32_t l = 1; l < FX_HEAD_LEVELS; ++l)
    if (l < h.n_levels && row >= h.lv[l].row0) v = h.lv[l];
  const uint32_t r = row - v.row0, cell = fx_fastdiv(r, v.anchors_magic, v.anchors_shift), a = r - cell * v.anchors;
  return (v.group0 + a * v.run_groups) * 256u + label * v.cells + cell;
}
// The decode of yolov3_bbox.py:12-23 with the operations of the region it stands for, one by one (nothing is contracted).
__device__ __forceinline__ float4 head_box(const HeadRow& r) {
  const float px = r.at[0], py = r.at[r.cells], pw = r.at[2u * (size_t)r.cells], ph = r.at[3u * (size_t)r.cells];
  const float4 b = make_float4(r.base[0], r.base[1], r.base[2], r.base[3]), s = make_float4(r.shift[0], r.shift[1], r.shift[2], r.shift[3]);
  const float stride = *r.stride;
  const float a0 = b.x + s.x, a1 = b.y + s.y, a2 = b.z + s.z, a3 = b.w + s.w;
  const float cx = (a0 + a2) * 0.5f + (fx_sigmoid(px) - 0.5f) * stride, cy = (a1 + a3) * 0.5f + (fx_sigmoid(py) - 0.5f) * stride;
  const float hw = (a2 - a0) * 0.5f * fx_exp(pw), hh = (a3 - a1) * 0.5f * fx_exp(ph);
  return make_float4(cx - hw, cy - hh, cx + hw, cy + hh);
}
__device__ __forceinline__ float head_objectness(const HeadRow& r) { return fx_sigmoid(r.at[4u * (size_t)r.cells]); }

// The scan of a head's class scores: elements that may pass the threshold go to LDS with their numbers.  They are compared as
// logits, with a bound below which none passes (launch): everything else is gather_own's, one element a thread, not a
// branch between the loads.  A workgroup with more of them than there is room for reads its share again and takes only those
// that are candidates.
// Four groups a wave in flight: with eight the kernel is larger, and its code takes longer to arrive than the loads save (12.0 us
// from the first workgroup's start to the last one's end of scan, 10.7 with four; 8.7 with the levels' arguments in one trip).
__device__ __forceinline__ void head_scan(const fx_nms_desc& d, const HeadMaps& h, const uint32_t key_cap, const uint32_t slices,
                                          const uint32_t task, const uint32_t slice, uint64_t* s_keys, uint32_t* s_count) {
  constexpr uint32_t U = 4u, WAVES = FX_NMS_THREADS / 64u;
  const uint32_t lane = threadIdx.x & 63u, wave = uni(threadIdx.x >> 6), C = d.n_classes;
  const uint32_t share = (h.groups + slices - 1u) / slices, first = min(slice * share, h.groups), end = min(first + share, h.groups);
  for (uint32_t pass = 0; pass < 2u; ++pass) {
    for (uint32_t g0 = first + wave; g0 < end; g0 += WAVES * U) {
      fx_u32x4_a4 v[U];
      uint32_t number[U], skip[U];   // skip: elements of the lane's four that are not its own (a run's last loads move back to its end)
#pragma unroll
      for (uint32_t u = 0; u < U; ++u) {
        const uint32_t g = uni(min(g0 + u * WAVES, end - 1u));
        HeadLevel lv = h.lv[0];   // (selects, not an index: the arguments come in one trip)
#pragma unroll
        for (uint32_t k = 1; k < FX_HEAD_LEVELS; ++k)
          if (k < h.n_levels && g >= h.lv[k].group0) lv = h.lv[k];
        const uint32_t a = fx_fastdiv(g - lv.group0, lv.run_magic, lv.run_shift), run0 = lv.group0 + a * lv.run_groups;
        const float* run = lv.map + ((size_t)(task * lv.anchors + a) * h.width + 5u) * lv.cells;
        const uint32_t own = (g - run0) * 256u + lane * 4u, from = min(own, C * lv.cells - 4u);
        v[u] = __builtin_nontemporal_load((const fx_u32x4_a4*)(run + from));   // (every line once)
        number[u] = run0 * 256u + from;
        skip[u] = g0 + u * WAVES < end ? own - from : 4u;
      }
      uint32_t mine = 0u;
#pragma unroll
      for (uint32_t u = 0; u < U; ++u)
#pragma unroll
        for (uint32_t e = 0; e < 4u; ++e)
          if (__uint_as_float(v[u][e]) >= h.logit_lo && e >= skip[u]) mine |= 1u << (u * 4u + e);
      if (mine == 0u) continue;
#pragma unroll
      for (uint32_t u = 0; u < U; ++u)
#pragma unroll
        for (uint32_t e = 0; e < 4u; ++e)
          if ((mine >> (u * 4u + e)) & 1u) {
            if (pass == 1u && !(fx_sigmoid(__uint_as_float(v[u][e])) > d.score_thr && head_objectness(head_row(h, task, number[u] + e)) >= h.keep_thr)) continue;
            const uint32_t slot = atomicAdd(s_count, 1u);
            if (slot < key_cap) s_keys[slot] = ((uint64_t)v[u][e] << 32) | (uint64_t)(number[u] + e);
          }
    }
    if (pass == 1u) break;
    __syncthreads();
    const bool again = *s_count > key_cap;
    __syncthreads();
    if (!again) break;
    if (threadIdx.x == 0u) *s_count = 0u;
    __syncthreads();
  }
}

// What a candidate needs besides its score is gathered here, by every workgroup for its own, one candidate a thread: a
// gather by the one that finishes the task is bound by the lines a CU gets (700 candidates of a head, seven lines each: 5.5 us),
// a gather in the scan sits between the rounds of loads.  Scores take their row's factor, a head's rows that are not kept
// leave, the largest coordinate goes to s_maxc, and the boxes to s_box where the candidates that are left are at most FX_NMS_FEW.
template <class Maps>
__device__ __forceinline__ void gather_own(const fx_nms_desc& d, const Maps& h, const uint32_t C, const uint32_t key_cap, const uint32_t task,
                                           const float* boxes, const float* factors, uint64_t* s_keys, float4* s_box, uint32_t* s_count,
                                           uint32_t* s_kept, uint32_t* s_maxc) {
  constexpr bool HEAD = !std::is_same_v<Maps, NoMaps>;
  const uint32_t n = min(*s_count, key_cap), over = *s_count - n;
  if (HEAD && threadIdx.x == 0u) *s_kept = 0u;
  if (HEAD) __syncthreads();
  // Where a head's scan found more than s_box holds, its memory is full of keys, of which the objectness may leave few: rows
  // first, then the boxes of what is left, from rows and labels (one 608 x 608 image, all of its 1.8 M scores above the
  // threshold, one row kept: the call 45 us, 62 with all boxes made, the chain of functors 57).
  const bool rows_first = HEAD && n > FX_NMS_FEW;
  uint32_t my_max = 0u;   // below orderable() of every value
  auto largest_of = [&](const float4& b) { my_max = max(my_max, max(max(orderable(b.x), orderable(b.y)), max(orderable(b.z), orderable(b.w)))); };
  for (uint32_t k0 = 0; k0 < n; k0 += FX_NMS_THREADS) {
    const uint32_t k = k0 + threadIdx.x;
    uint64_t key = 0ull;
    float4 b = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    bool keep = k < n;
    if (keep) {
      key = s_keys[k];
      float f = 1.0f;
      if constexpr (HEAD) {
        const HeadRow r = head_row(h, task, (uint32_t)key);
        const float score = fx_sigmoid(__uint_as_float((uint32_t)(key >> 32)));
        f = head_objectness(r);
        if (!rows_first) b = head_box(r);
        keep = score > d.score_thr && f >= h.keep_thr;
        key = ((uint64_t)(~orderable(score)) << 32) | (uint64_t)(r.row * C + r.label);
      } else {
        const uint32_t r = (uint32_t)key / C;
        if (factors) f = factors[r];
        b = *(const float4*)(boxes + (size_t)r * 4u);
      }
      if (HEAD || factors) key = ((uint64_t)(~orderable(from_orderable(~(uint32_t)(key >> 32)) * f)) << 32) | (uint64_t)(uint32_t)key;
      if (keep && !rows_first) largest_of(b);
    }
    if (HEAD) __syncthreads();   // (the places that are written lie among those that have been read)
    if (keep) {
      const uint32_t at = HEAD ? atomicAdd(s_kept, 1u) : k;
      if (HEAD || factors) s_keys[at] = key;
      if (n <= FX_NMS_FEW && key_cap >= FX_NMS_ROOMY) s_box[at] = b;
    }
  }
  if constexpr (HEAD) {
    if (rows_first) {
      __syncthreads();
      const uint32_t kept = *s_kept;
      for (uint32_t k = threadIdx.x; k < kept; k += FX_NMS_THREADS) {
        const uint32_t idx = (uint32_t)s_keys[k], r = fx_fastdiv(idx, h.c_magic, h.c_shift);
        const float4 b = head_box(head_row(h, task, head_number(h, r, idx - r * C)));
        largest_of(b);
        if (kept <= FX_NMS_FEW && key_cap >= FX_NMS_ROOMY) s_box[k] = b;
      }
    }
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) my_max = max(my_max, (uint32_t)__shfl_xor((int)my_max, o, 64));
  if ((threadIdx.x & 63u) == 0u && my_max != 0u) atomicMax(s_maxc, my_max);
  __syncthreads();
  if (HEAD) {
    if (threadIdx.x == 0u) *s_count = *s_kept + over;
    __syncthreads();
  }
}

// Maps: NoMaps (boxes and scores as the descriptor has them) or HeadMaps (rows that the kernel takes from a head's maps itself).
template <class Maps>
__global__ __launch_bounds__(FX_NMS_THREADS) void fx_sort_nms_kernel(const fx_nms_desc d, const Maps h, const uint32_t key_cap,
                                                                    const uint32_t slices, uint32_t* const ws,
                                                                    uint32_t* err_host) {
  constexpr bool HEAD = !std::is_same_v<Maps, NoMaps>;
  extern __shared__ __attribute__((aligned(16))) uint64_t s_keys[];   // key_cap (a power of two)
  __shared__ float4 s_kbox[FX_NMS_MAX_OUT];
  __shared__ float s_karea[FX_NMS_MAX_OUT];
  __shared__ uint32_t s_kept[FX_NMS_MAX_OUT];   // places in score order
  __shared__ float4 s_cbox[FX_NMS_CHUNK];       // chunk: original boxes
  __shared__ float4 s_obox[FX_NMS_CHUNK];       // chunk: boxes moved by their class offset
  __shared__ float s_carea[FX_NMS_CHUNK];
  __shared__ uint32_t s_clabel[FX_NMS_CHUNK];
  __shared__ uint32_t s_in[2][FX_NMS_CHUNK][2]; // by the chunk's parity: earlier candidates of the chunk that overlap candidate j
  __shared__ uint32_t s_dead[2][2];             // candidates of the chunk that the kept list overlaps
  __shared__ uint32_t s_count, s_maxc, s_nk, s_base, s_ticket;
  __shared__ uint32_t s_lo, s_hi, s_crowd, s_wave[FX_NMS_THREADS / 64u];

  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const uint32_t task = blockIdx.x / slices, slice = blockIdx.x - task * slices;
  uint32_t* const ctr = ws + (size_t)task * FX_NMS_WS_WORDS;   // [0] candidates, [1] finished slices, [2] largest coordinate
  uint64_t* const g_keys = (uint64_t*)(ws + (size_t)d.n_tasks * FX_NMS_WS_WORDS) + (size_t)task * key_cap;
  const bool roomy = key_cap >= FX_NMS_ROOMY;
  uint64_t* const g_box = (uint64_t*)(ws + (size_t)d.n_tasks * FX_NMS_WS_WORDS) + (size_t)d.n_tasks * key_cap + (size_t)task * (2u * FX_NMS_FEW);
  // NC classes, in rows of C elements (C > NC: columns behind the class scores that are not candidates)
  const uint32_t NC = d.mode == 1 ? d.n_classes : 1u;
  const uint32_t C = (d.mode == 1 && d.scores_row_stride != 0u) ? d.scores_row_stride : NC;
  const float* boxes = d.boxes + (int64_t)task * d.boxes_task_stride;
  const float* scores = d.scores + (int64_t)task * d.scores_task_stride;
  const float* factors = d.factors ? d.factors + (int64_t)task * d.factors_task_stride : nullptr;
  const int64_t* labels = d.labels ? d.labels + (int64_t)task * d.labels_task_stride : nullptr;
  float* dets = d.dets + (size_t)task * d.max_num * 5u;
  int64_t* out_labels = d.out_labels + (size_t)task * d.max_num;
  int64_t* out_index = d.out_index ? d.out_index + (size_t)task * d.max_num : nullptr;

  if (tid == 0) {
    s_count = 0u;
    s_maxc = 0u;
  }
  uint32_t rows = d.rows;
  if constexpr (!HEAD) {
    // The task's row count may lie in host memory, where a read costs a trip over the bus and the
    // reads of many workgroups queue up: slice 0 reads it and passes it on through the workspace
    // (count + 1 in ctr[3]); a slice that does not see it within its polls reads it itself.
    if (tid == 0) {
      if (d.counts) {
        uint32_t seen = 0u;
        if (slice != 0u)
          for (uint32_t polls = 0; polls < 4096u && seen == 0u; ++polls) {
            seen = __hip_atomic_load(&ctr[3], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (seen == 0u) __builtin_amdgcn_s_sleep(2);
          }
        if (seen == 0u) {
          seen = min(d.rows, __hip_atomic_load(d.counts + task, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM)) + 1u;
          if (slice == 0u) __hip_atomic_store(&ctr[3], seen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        rows = seen - 1u;
      }
      s_base = rows;
    }
    __syncthreads();
    rows = s_base;
  }
  __syncthreads();   // s_base is used again below

  FX_NMS_STAMP(0);
  if constexpr (HEAD) {
    head_scan(d, h, key_cap, slices, task, slice, s_keys, &s_count);
  } else {
    // 1. candidates: four 128-bit loads per thread in flight
    const uint32_t all_items = rows * C;   // < 2^32 (host)
    // this workgroup's share: a multiple of four items, so that its 128-bit loads stay aligned
    const uint32_t share = (((all_items + slices - 1u) / slices) + 3u) & ~3u;
    const uint32_t first = min(slice * share, all_items);
    const uint32_t n_items = min(first + share, all_items);   // end of the share
    const bool vec = (((uintptr_t)scores) & 15u) == 0u;
    constexpr uint32_t U = 4u, PER_ROUND = FX_NMS_THREADS * U * 4u;
    for (uint32_t base = first; base < n_items; base += PER_ROUND) {
      float v[U][4];
  #pragma unroll
      for (uint32_t u = 0; u < U; ++u) {
        const uint32_t i0 = base + (u * FX_NMS_THREADS + tid) * 4u;
        if (vec && i0 + 3u < n_items) {
          const float4 q = *(const float4*)(scores + i0);
          v[u][0] = q.x; v[u][1] = q.y; v[u][2] = q.z; v[u][3] = q.w;
        } else {
  #pragma unroll
          for (uint32_t e = 0; e < 4u; ++e) v[u][e] = i0 + e < n_items ? scores[i0 + e] : d.score_thr;   // the threshold itself never passes
        }
      }
      uint32_t mine = 0u;   // bit u * 4 + e: element passes
  #pragma unroll
      for (uint32_t u = 0; u < U; ++u)
  #pragma unroll
        for (uint32_t e = 0; e < 4u; ++e)
          if (v[u][e] > d.score_thr) mine |= 1u << (u * 4u + e);
      // few elements pass a detector's threshold: a lane that has some takes its places with one LDS
      // atomic (the order of arrival does not matter), the others go straight on to the next loads
      if (mine == 0u) continue;
      if (C != NC) {   // columns behind the class scores are no candidates
  #pragma unroll
        for (uint32_t u = 0; u < U; ++u)
  #pragma unroll
          for (uint32_t e = 0; e < 4u; ++e)
            if (((mine >> (u * 4u + e)) & 1u) && (base + (u * FX_NMS_THREADS + tid) * 4u + e) % C >= NC) mine &= ~(1u << (u * 4u + e));
        if (mine == 0u) continue;
      }
      uint32_t slot = atomicAdd(&s_count, (uint32_t)__popc(mine));
  #pragma unroll
      for (uint32_t u = 0; u < U; ++u)
  #pragma unroll
        for (uint32_t e = 0; e < 4u; ++e) {
          if ((mine >> (u * 4u + e)) & 1u) {
            const uint32_t i = base + (u * FX_NMS_THREADS + tid) * 4u + e;
            // (the raw score for now: gather_own applies the row's factor)
            if (slot < key_cap) s_keys[slot] = ((uint64_t)(~orderable(v[u][e])) << 32) | (uint64_t)i;
            ++slot;
          }
        }
    }
  }
  __syncthreads();
  FX_NMS_STAMP(1);
  float4* const s_own = (float4*)(s_keys + FX_NMS_FEW);   // (with FX_NMS_ROOMY)
  gather_own(d, h, C, key_cap, task, boxes, d.mode == 1 ? factors : nullptr, s_keys, s_own, &s_count, &s_base, &s_maxc);
  uint64_t key[FX_NMS_OWN], corner[FX_NMS_OWN][2];
  uint32_t count, largest;
  if (slices > 1u) {
    // hand this workgroup's keys over and take a ticket
    const uint32_t mine = min(s_count, key_cap);
    if (tid == 0) {
      s_base = atomicAdd(&ctr[0], s_count);
      if (mine != 0u) atomicMax(&ctr[2], s_maxc);
    }
    __syncthreads();
    const uint32_t gbase = s_base;
    // Keys and counters are written with device-scope atomic accesses, which go through to the
    // memory side of the caches, and the ticket is taken only after they have been acknowledged:
    // no release / acquire fence, which on this device would write back and invalidate whole
    // caches once per workgroup.  This rests on the device: a relaxed device-scope store is
    // performed at the memory side of the caches by the time it is acknowledged (vmcnt).  The
    // compiler is told the order explicitly: nothing moves across the signal fences.
    for (uint32_t k = tid; k < mine; k += FX_NMS_THREADS)
      if (gbase + k < key_cap) __hip_atomic_store(&g_keys[gbase + k], s_keys[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (roomy)   // (a workgroup that keeps more candidates than that has no boxes: neither has the task need of any)
      for (uint32_t k = tid; k < 2u * mine && (k >> 1) + gbase < FX_NMS_FEW; k += FX_NMS_THREADS)
        if (mine <= FX_NMS_FEW) __hip_atomic_store(&g_box[2u * gbase + k], ((const uint64_t*)s_own)[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __syncthreads();
    if (tid == 0) s_ticket = atomicAdd(&ctr[1], 1u);
    __syncthreads();
    if (s_ticket != slices - 1u) return;   // somebody else finishes the task
    FX_NMS_STAMP(2);
    // the last workgroup of the task: everything the others wrote is visible.  The first candidates are asked for
    // together with their number.
#pragma unroll
    for (uint32_t i = 0; i < FX_NMS_OWN; ++i) {
      const uint32_t k = i * FX_NMS_THREADS + tid;
      key[i] = __hip_atomic_load(&g_keys[min(k, key_cap - 1u)], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      corner[i][0] = corner[i][1] = 0ull;
      if (roomy) {
        corner[i][0] = __hip_atomic_load(&g_box[2u * k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        corner[i][1] = __hip_atomic_load(&g_box[2u * k + 1u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    count = uni(__hip_atomic_load(&ctr[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    largest = __hip_atomic_load(&ctr[2], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  } else {
    // the only one: its own candidates are all
    count = uni(s_count);
    largest = s_maxc;
#pragma unroll
    for (uint32_t i = 0; i < FX_NMS_OWN; ++i) {
      const uint32_t k = i * FX_NMS_THREADS + tid;
      key[i] = 0ull;
      corner[i][0] = corner[i][1] = 0ull;
      if (!roomy || count > FX_NMS_FEW || k >= count) continue;
      key[i] = s_keys[k];
      corner[i][0] = ((const uint64_t*)s_own)[2u * k];
      corner[i][1] = ((const uint64_t*)s_own)[2u * k + 1u];
    }
  }
  const float class_step = from_orderable(largest) + 1.0f;   // (no candidates: not used)
  if (tid == 0) {
    s_lo = ~0u;
    s_hi = 0u;
    s_crowd = 0u;
  }
  __syncthreads();
  if (tid == 0) {   // the counters are zero again for the next launch
    __hip_atomic_store(&ctr[0], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&ctr[1], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&ctr[2], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&ctr[3], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (count > key_cap) {   // more candidates than the launch was sized for: reported, nothing returned
    if (tid == 0) {
      // (a host that polls n_out takes the report back when it sees the overflow: the report has to be there by then)
      if (err_host) __hip_atomic_store(err_host, (uint32_t)FX_ASYNC_NMS_CAPACITY, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      __hip_atomic_store(d.n_out + task, FX_NMS_OVERFLOW, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    for (uint32_t k = tid; k < d.max_num * 5u; k += FX_NMS_THREADS) dets[k] = 0.0f;
    for (uint32_t k = tid; k < d.max_num; k += FX_NMS_THREADS) {
      out_labels[k] = 0;
      if (out_index) out_index[k] = 0;
    }
    return;
  }
  // what a key stands for
  auto row_of = [&](uint32_t idx) { return HEAD ? fx_fastdiv(idx, divisor_magic(h), divisor_shift(h)) : idx / C; };
  auto label_of = [&](uint32_t idx, uint32_t r) { return d.mode == 1 ? idx - r * C : (labels ? (uint32_t)labels[idx] : 0u); };
  auto moved_by = [](const float4& b, float off) { return make_float4(b.x + off, b.y + off, b.z + off, b.w + off); };
  auto area_of = [](const float4& b) { return (b.z - b.x) * (b.w - b.y); };

  // Of up to FX_NMS_OWN candidates a thread, everything the walk needs lies in LDS in score order (s_keys' memory, whose
  // keys have been handed over): buckets, keys by bucket, keys in order, moved boxes, boxes, areas, labels.
  const uint32_t np = (count + 63u) & ~63u;
  uint32_t* const s_bucket = (uint32_t*)s_keys;
  uint64_t* const s_part = (uint64_t*)(s_bucket + FX_NMS_BUCKETS);
  uint64_t* const s_order = s_part + np;
  float4* const s_moved = (float4*)(s_order + np);
  float4* const s_box = s_moved + np;
  float* const s_area = (float*)(s_box + np);
  uint32_t* const s_label = (uint32_t*)(s_area + np);
  bool placed = roomy && count <= FX_NMS_FEW;
  FX_NMS_STAMP(3);
  if (placed) {
    // 2. order by buckets of the score's bits: a candidate's bucket says how many lie ahead of it but for its
    // bucket's own, of which there are one or two (700 candidates, 2 048 buckets between the lowest score and the highest).
    uint32_t label[FX_NMS_OWN], lo = ~0u, hi = 0u;
#pragma unroll
    for (uint32_t i = 0; i < FX_NMS_BUCKETS / FX_NMS_THREADS; ++i) s_bucket[i * FX_NMS_THREADS + tid] = 0u;
#pragma unroll
    for (uint32_t i = 0; i < FX_NMS_OWN; ++i) {
      label[i] = 0u;
      if (i * FX_NMS_THREADS + tid >= count) continue;
      const uint32_t idx = (uint32_t)key[i];
      label[i] = label_of(idx, row_of(idx));
      lo = min(lo, (uint32_t)(key[i] >> 32));
      hi = max(hi, (uint32_t)(key[i] >> 32));
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
      lo = min(lo, (uint32_t)__shfl_xor((int)lo, o, 64));
      hi = max(hi, (uint32_t)__shfl_xor((int)hi, o, 64));
    }
    if (lane == 0u && lo <= hi) {
      atomicMin(&s_lo, lo);
      atomicMax(&s_hi, hi);
    }
    __syncthreads();
    const uint32_t first = uni(s_lo), range = uni(s_hi) - first;
    const uint32_t shift = range < FX_NMS_BUCKETS ? 0u : 32u - (uint32_t)__builtin_clz(range) - FX_NMS_BUCKET_BITS;
    uint32_t bucket[FX_NMS_OWN], slot[FX_NMS_OWN];
#pragma unroll
    for (uint32_t i = 0; i < FX_NMS_OWN; ++i) {
      bucket[i] = 0u;
      if (i * FX_NMS_THREADS + tid >= count) continue;
      bucket[i] = ((uint32_t)(key[i] >> 32) - first) >> shift;
      slot[i] = atomicAdd(&s_bucket[bucket[i]], 1u);
    }
    __syncthreads();
    {
      const uint2 n = ((const uint2*)s_bucket)[tid];
      static_assert(FX_NMS_BUCKETS == 2u * FX_NMS_THREADS, "two buckets a thread");
      uint32_t ahead = n.x + n.y;
#pragma unroll
      for (uint32_t o = 1; o < 64u; o <<= 1) {
        const uint32_t t = (uint32_t)__shfl_up((int)ahead, o, 64);
        ahead += lane >= o ? t : 0u;
      }
      if (lane == 63u) s_wave[wave] = ahead;
      if (max(n.x, n.y) > FX_NMS_CROWD) s_crowd = 1u;
      __syncthreads();
      const uint32_t w = s_wave[lane & (FX_NMS_THREADS / 64u - 1u)];
      ahead += fx_wave_sum(lane < wave ? w : 0u, lane) - n.x - n.y;
      ((uint2*)s_bucket)[tid] = make_uint2(ahead | (n.x << 16), (ahead + n.x) | (n.y << 16));   // start and number
    }
    placed = uni(s_crowd) == 0u;   // many scores in one bucket (all alike, say): the sort below
    __syncthreads();
    if (placed) {
      uint32_t entry[FX_NMS_OWN];
#pragma unroll
      for (uint32_t i = 0; i < FX_NMS_OWN; ++i) {
        if (i * FX_NMS_THREADS + tid >= count) continue;
        entry[i] = s_bucket[bucket[i]];
        s_part[(entry[i] & 0xffffu) + slot[i]] = key[i];
      }
      __syncthreads();
#pragma unroll
      for (uint32_t i = 0; i < FX_NMS_OWN; ++i) {
        if (i * FX_NMS_THREADS + tid >= count) continue;
        const uint32_t start = entry[i] & 0xffffu, n = entry[i] >> 16;
        uint32_t at = start;
        if (n > 1u)
          for (uint32_t k = 0; k < n; ++k) at += s_part[start + k] < key[i] ? 1u : 0u;
        const float4 b = make_float4(__uint_as_float((uint32_t)corner[i][0]), __uint_as_float((uint32_t)(corner[i][0] >> 32)),
                                     __uint_as_float((uint32_t)corner[i][1]), __uint_as_float((uint32_t)(corner[i][1] >> 32)));
        const float4 m = moved_by(b, (float)label[i] * class_step);
        s_order[at] = key[i];
        s_moved[at] = m;
        s_box[at] = b;
        s_area[at] = area_of(m);
        s_label[at] = label[i];
      }
      FX_NMS_STAMP(4);
    } else {
#pragma unroll
      for (uint32_t i = 0; i < FX_NMS_OWN; ++i)
        if (i * FX_NMS_THREADS + tid < count) s_keys[i * FX_NMS_THREADS + tid] = key[i];
    }
  } else {
    if (slices > 1u)
      for (uint32_t k = tid; k < count; k += FX_NMS_THREADS) s_keys[k] = __hip_atomic_load(&g_keys[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (!placed) {
    // 2. bitonic sort (ascending keys = descending score, ascending index); the tail is padding.
    // Stages whose partners lie at most 64 apart stay inside aligned blocks of 128 keys: a wave
    // runs all of them on its blocks without a workgroup barrier (LDS accesses of one wave are
    // performed in order), so a phase costs one barrier per wider stage plus one.
    uint32_t n2 = 128u;
    while (n2 < count) n2 <<= 1;
    for (uint32_t i = count + tid; i < n2; i += FX_NMS_THREADS) s_keys[i] = ~0ull;
    __syncthreads();
    auto exchange = [&](uint32_t i, uint32_t j, uint32_t k) {
      const uint32_t l = i | j;
      const uint64_t a = s_keys[i], b = s_keys[l];
      const bool up = (i & k) == 0u;
      if ((a > b) == up) { s_keys[i] = b; s_keys[l] = a; }
    };
    auto narrow_stages = [&](uint32_t k_first, uint32_t k_last) {   // every stage j <= 64 of phases k_first .. k_last
      for (uint32_t blk = wave; blk < (n2 >> 7); blk += FX_NMS_THREADS / 64u) {
        // the block's 128 keys in registers, two a lane (positions lane and lane + 64): the stages
        // exchange them between lanes, LDS is read and written once per call
        const uint32_t p0 = (blk << 7) + lane;
        uint64_t ka = s_keys[p0], kb = s_keys[p0 + 64u];
        for (uint32_t k = k_first; k <= k_last; k <<= 1) {
          const bool up_a = (p0 & k) == 0u, up_b = ((p0 + 64u) & k) == 0u;
          if (k >= 128u) {   // partners 64 apart: the lane's own two keys (up_a == up_b here)
            const bool sw = (ka > kb) == up_a;
            const uint64_t lo = sw ? kb : ka, hi = sw ? ka : kb;
            ka = lo; kb = hi;
          }
          if (k >= 64u) { ka = bitonic_step<32>(ka, up_a, lane); kb = bitonic_step<32>(kb, up_b, lane); }
          if (k >= 32u) { ka = bitonic_step<16>(ka, up_a, lane); kb = bitonic_step<16>(kb, up_b, lane); }
          if (k >= 16u) { ka = bitonic_step<8>(ka, up_a, lane); kb = bitonic_step<8>(kb, up_b, lane); }
          if (k >= 8u) { ka = bitonic_step<4>(ka, up_a, lane); kb = bitonic_step<4>(kb, up_b, lane); }
          if (k >= 4u) { ka = bitonic_step<2>(ka, up_a, lane); kb = bitonic_step<2>(kb, up_b, lane); }
          ka = bitonic_step<1>(ka, up_a, lane); kb = bitonic_step<1>(kb, up_b, lane);
        }
        s_keys[p0] = ka; s_keys[p0 + 64u] = kb;
      }
    };
    narrow_stages(2u, 128u);
    __syncthreads();
    for (uint32_t k = 256u; k <= n2; k <<= 1) {
      for (uint32_t j = k >> 1; j >= 128u; j >>= 1) {
        for (uint32_t p = tid; p < (n2 >> 1); p += FX_NMS_THREADS) exchange(((p & ~(j - 1u)) << 1) | (p & (j - 1u)), j, k);
        __syncthreads();
      }
      narrow_stages(k, k);
      __syncthreads();
    }
    FX_NMS_STAMP(4);
  }

  auto write_out = [&](uint32_t slot, uint64_t k, const float4& b, uint32_t label) {
    float* o = dets + (size_t)slot * 5u;
    o[0] = b.x; o[1] = b.y; o[2] = b.z; o[3] = b.w;
    o[4] = from_orderable(~(uint32_t)(k >> 32));
    out_labels[slot] = (int64_t)label;
    if (out_index) out_index[slot] = (int64_t)(d.mode == 1 ? row_of((uint32_t)k) * NC + label : (uint32_t)k);   // position among the candidates proper
  };

  // 3. greedy walk
  if (tid == 0) s_nk = 0u;
  if (tid < 4u * FX_NMS_CHUNK) ((uint32_t*)s_in)[tid] = 0u;
  if (tid < 4u) ((uint32_t*)s_dead)[tid] = 0u;
  __syncthreads();
  uint32_t nk = 0u, p = 0u;
  // (not placed: boxes of a chunk are asked for while the one before is decided)
  float4 next = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  uint32_t next_label = 0u;
  auto ask = [&](uint32_t pos) {
    if (tid >= FX_NMS_CHUNK || pos + tid >= count) return;
    const uint32_t idx = (uint32_t)s_keys[pos + tid], r = row_of(idx);
    next_label = label_of(idx, r);
    if constexpr (HEAD) next = head_box(head_row(h, task, head_number(h, r, next_label)));
    else next = *(const float4*)(boxes + (size_t)r * 4u);
  };
  if (!placed) ask(0u);
  for (uint32_t pos = 0; pos < count && nk < d.max_num; pos += FX_NMS_CHUNK, p ^= 1u) {
    const uint32_t m = min(FX_NMS_CHUNK, count - pos);
    if (!placed) {
      if (tid < m) {
        const float4 q = moved_by(next, (float)next_label * class_step);
        s_cbox[tid] = next;
        s_obox[tid] = q;
        s_carea[tid] = area_of(q);
        s_clabel[tid] = next_label;
      }
      __syncthreads();
      ask(pos + FX_NMS_CHUNK);
    }
    const float4* const moved = placed ? s_moved + pos : s_obox;
    const float* const areas = placed ? s_area + pos : s_carea;
    if (nk != 0u) {
      // candidate `lane` against every 16th kept box, four of them at a time (a box that is there twice does not matter)
      const float4 q = moved[min(lane, m - 1u)];
      const float ca = areas[min(lane, m - 1u)];
      uint64_t dead = 0ull;
      for (uint32_t k = uni(wave); k < nk; k += FX_NMS_THREADS / 16u) {
        float4 o[4];
        float oa[4];
        uint64_t near[4];
#pragma unroll
        for (uint32_t e = 0; e < 4u; ++e) {
          o[e] = s_kbox[min(k + e * (FX_NMS_THREADS / 64u), nk - 1u)];
          oa[e] = s_karea[min(k + e * (FX_NMS_THREADS / 64u), nk - 1u)];
        }
#pragma unroll
        for (uint32_t e = 0; e < 4u; ++e) near[e] = near_lanes(o[e], q, d.iou_thr) & ~dead;
        if ((near[0] | near[1] | near[2] | near[3]) == 0ull) continue;
#pragma unroll
        for (uint32_t e = 0; e < 4u; ++e)
          if (near[e] != 0ull) dead |= overlap_lanes(near[e], o[e], oa[e], q, ca, d.iou_thr);
      }
      if (dead != 0ull && lane < 2u) atomicOr(&s_dead[p][lane], (uint32_t)(dead >> (32u * lane)));
      __syncthreads();
    }
    {
      // inside the chunk: pairs (i, j), i < j, of candidates that no kept box overlaps; lanes behind i take (i, lane), those
      // before it (63 - i, 63 - lane), so that two rows of pairs fill one wave
      const uint64_t gone = ((uint64_t)uni(s_dead[p][1]) << 32) | (uint64_t)uni(s_dead[p][0]);
#pragma unroll
      for (uint32_t e = 0; e < 2u; ++e) {
        const uint32_t row = uni(wave) * 2u + e, other = 63u - row;
        if (((gone >> row) & (gone >> other) & 1ull) != 0ull) continue;
        const bool back = lane < row;
        const uint32_t pi = back ? other : row, pj = back ? 63u - lane : lane, i = min(pi, m - 1u), j = min(pj, m - 1u);   // (pairs that are none: not looked at below)
        const float4 bi = moved[i], bj = moved[j];
        const float ai = areas[i], aj = areas[j];
        const uint64_t pairs = __ballot(pi < pj && pj < m && ((gone >> pi) & 1ull) == 0ull && ((gone >> pj) & 1ull) == 0ull);
        const uint64_t near = near_lanes(bi, bj, d.iou_thr) & pairs;
        if (near == 0ull) continue;
        const uint64_t over = overlap_lanes(near, bi, ai, bj, aj, d.iou_thr);
        if (((over >> lane) & 1ull) != 0ull) atomicOr(&s_in[p][pj][pi >> 5], 1u << (pi & 31u));
      }
    }
    __syncthreads();
    if (wave == 1u) {   // for the chunk after this one; the last to read these has passed a barrier
      s_in[p ^ 1u][lane][0] = 0u;
      s_in[p ^ 1u][lane][1] = 0u;
      if (lane < 2u) s_dead[p ^ 1u][lane] = 0u;
    }
    if (wave == 0u) {
      // In order, candidate i is kept unless a kept one before it overlaps it.  All candidates
      // decide together, round after round: one with a kept overlapping predecessor is dead, one
      // whose overlapping predecessors are all dead is kept, the others wait; the first undecided
      // candidate always decides, and with few overlaps two or three rounds settle the chunk
      // (a walk from candidate to candidate costs 64 dependent steps).
      const uint64_t in = ((uint64_t)s_in[p][lane][1] << 32) | (uint64_t)s_in[p][lane][0];
      const uint64_t valid = m >= 64u ? ~0ull : (1ull << m) - 1ull;
      uint64_t deadm = (((uint64_t)uni(s_dead[p][1]) << 32) | (uint64_t)uni(s_dead[p][0])) | ~valid;
      uint64_t keptm = 0ull;
      bool decided = ((deadm >> lane) & 1ull) != 0ull;
      for (;;) {
        const bool now_dead = !decided && (in & keptm) != 0ull;
        const bool now_kept = !decided && !now_dead && (in & ~deadm) == 0ull;
        const uint64_t nd = __ballot(now_dead), nkp = __ballot(now_kept);
        if ((nd | nkp) == 0ull) break;
        deadm |= nd;
        keptm |= nkp;
        decided = decided || now_dead || now_kept;
      }
      // the walk ends when max_num are kept: the first `room` of them in order
      const uint32_t room = d.max_num - nk;
      const uint32_t rank = (uint32_t)__popcll(keptm & ((1ull << lane) - 1ull));
      const uint64_t keep = __ballot(((keptm >> lane) & 1ull) != 0ull && rank < room);
      const uint32_t kept_now = (uint32_t)__popcll(keep);
      if ((keep >> lane) & 1ull) {
        const uint32_t slot = nk + rank;
        s_kbox[slot] = moved[lane];
        s_karea[slot] = areas[lane];
        s_kept[slot] = pos + lane;
        if (!placed) write_out(slot, s_keys[pos + lane], s_cbox[lane], s_clabel[lane]);
      }
      if (lane == 0u) s_nk = nk + kept_now;
    }
    __syncthreads();
    nk = uni(s_nk);
  }
  FX_NMS_STAMP(5);
  // (behind the walk, not in it: its barriers would wait until the stores have been acknowledged)
  if (placed)
    for (uint32_t k = tid; k < nk; k += FX_NMS_THREADS) write_out(k, s_order[s_kept[k]], s_box[s_kept[k]], s_label[s_kept[k]]);
  // rows past the kept ones are zero: the outputs have a fixed shape
  for (uint32_t k = nk * 5u + tid; k < d.max_num * 5u; k += FX_NMS_THREADS) dets[k] = 0.0f;
  for (uint32_t k = nk + tid; k < d.max_num; k += FX_NMS_THREADS) {
    out_labels[k] = 0;
    if (out_index) out_index[k] = 0;
  }
  // (system scope: a count in pinned host memory goes through to the host, which may be polling it)
  if (tid == 0) __hip_atomic_store(d.n_out + task, nk, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace

static uint32_t device_cus() {
  static int cus = 0;
  if (cus == 0) {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) == hipSuccess && hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0) cus = n;
    else cus = 256;
  }
  return (uint32_t)cus;
}

// slices of a task: a workgroup per CU over all tasks (a CU takes one workgroup of 1024 threads at
// a time: with two per CU the second half of the launch starts when the first ends, 16 us into
// the kernel for 16 images), none with less than one round of loads
uint32_t fx_nms_slices(const fx_nms_desc& d) {
  const uint64_t items = (uint64_t)d.rows * (d.mode == 1 ? std::max(d.n_classes, d.scores_row_stride) : 1u);
  const uint64_t per_round = (uint64_t)FX_NMS_THREADS * 16u;
  uint64_t s = (items + per_round - 1) / per_round;
  const uint64_t want = d.n_tasks > 0 ? std::max<uint32_t>(device_cus() / (uint32_t)d.n_tasks, 1u) : 1u;
  if (s > want) s = want;
  if (s > 64) s = 64;
  return s < 1 ? 1u : (uint32_t)s;
}

size_t fx_nms_workspace_bytes(int n_tasks, uint32_t key_cap) {
  return (size_t)n_tasks * ((size_t)FX_NMS_WS_WORDS * 4 + (size_t)key_cap * 8 + (key_cap >= FX_NMS_ROOMY ? FX_NMS_FEW * 16u : 0u));
}
size_t fx_nms_workspace_clear_bytes(int n_tasks) { return (size_t)n_tasks * FX_NMS_WS_WORDS * 4; }

// 0: launched; otherwise a HIP error code + 100
template <class Maps>
static int launch_sort_nms(const fx_nms_desc& d, const Maps& maps, uint32_t slices, uint32_t key_cap, void* workspace, uint32_t* err_host,
                           hipStream_t stream) {
  const size_t lds = (size_t)key_cap * sizeof(uint64_t);
  hipError_t e = hipSuccess;
  if (lds > 32768) {   // beyond what a kernel gets without asking: raised once per device, to the most a launch may need
    static std::mutex mu;
    static bool raised[64] = {};
    int dev = 0;
    e = hipGetDevice(&dev);
    if (e != hipSuccess) return 100 + (int)e;
    std::lock_guard<std::mutex> lock(mu);
    if (dev < 0 || dev >= 64 || !raised[dev]) {
      e = hipFuncSetAttribute((const void*)fx_sort_nms_kernel<Maps>, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)(FX_NMS_MAX_CANDIDATES * sizeof(uint64_t)));
      if (e != hipSuccess) return 100 + (int)e;
      if (dev >= 0 && dev < 64) raised[dev] = true;
    }
  }
  hipLaunchKernelGGL(fx_sort_nms_kernel<Maps>, dim3((uint32_t)d.n_tasks * slices), dim3(FX_NMS_THREADS), lds, stream, d, maps, key_cap,
                     slices, (uint32_t*)workspace, err_host);
  e = hipGetLastError();
  return e == hipSuccess ? 0 : 100 + (int)e;
}

int fx_launch_sort_nms(const fx_nms_desc& d, uint32_t key_cap, void* workspace, uint32_t* err_host, hipStream_t stream) {
  return launch_sort_nms(d, NoMaps{}, fx_nms_slices(d), key_cap, workspace, err_host, stream);
}

// no logit below it has a score above thr (the device's sigmoid is off by less than 1e-6, so nothing up to the logit of
// thr less 1e-5 of it passes; a threshold of 1 or more, or NaN, lets nothing pass, and one below 0 every number, with -inf,
// whose score is 0: the bound itself is one of the logits that are looked at)
static float logit_bound(float thr) {
  const double t = (double)thr * (1.0 - 1e-5);
  if (!(thr < 1.0f)) return std::numeric_limits<float>::infinity();
  if (!(t > 1e-30)) return thr < 0.0f ? -std::numeric_limits<float>::infinity() : std::numeric_limits<float>::lowest();
  const double x = std::log(t / (1.0 - t));
  return std::nextafterf((float)x, -std::numeric_limits<float>::infinity());
}

int fx_launch_head_nms(const fx_head_desc& head, const fx_nms_desc& d, uint32_t key_cap, void* workspace, uint32_t* err_host, hipStream_t stream) {
  HeadMaps m;
  memset(&m, 0, sizeof m);
  m.n_levels = (uint32_t)head.n_levels;
  m.width = 5u + d.n_classes;
  m.keep_thr = head.keep_thr;
  m.logit_lo = logit_bound(d.score_thr);
  m.strides = head.strides;
  fx_fastdiv_make(d.n_classes, &m.c_magic, &m.c_shift);
  uint32_t rows = 0u;
  for (int l = 0; l < head.n_levels; ++l) {
    HeadLevel& v = m.lv[l];
    v.map = head.maps[l];
    v.base = head.bases[l];
    v.shift = head.shifts[l];
    v.cells = head.cells[l];
    v.anchors = head.anchors[l];
    v.row0 = rows;
    v.group0 = m.groups;
    v.run_groups = (d.n_classes * v.cells + 255u) / 256u;
    fx_fastdiv_make(v.cells, &v.cells_magic, &v.cells_shift);
    fx_fastdiv_make(v.run_groups, &v.run_magic, &v.run_shift);
    fx_fastdiv_make(v.anchors, &v.anchors_magic, &v.anchors_shift);
    rows += v.cells * v.anchors;
    m.groups += v.run_groups * v.anchors;
  }
  // a workgroup per CU over all images, at most 128 an image (above HeadLevel), none without a group for every wave
  const uint32_t slices = std::min<uint32_t>(std::min<uint32_t>(std::max(device_cus() / (uint32_t)d.n_tasks, 1u), 128u),
                                             (m.groups + FX_NMS_THREADS / 64u - 1u) / (FX_NMS_THREADS / 64u));
  return launch_sort_nms(d, m, slices, key_cap, workspace, err_host, stream);
}
