// Hand-written kernel for one region shape: the decode + score filter of a YOLO-style detection
// head (functs/benchmark/ai_model/yolov3/yolov3_bbox.py:12-23, 104-130 in the reference: sigmoid
// of the centre offsets, exp of the sizes, anchors and strides, objectness threshold, kept rows
// of boxes / class scores / objectness).  A plan whose lowered programs ARE that computation
// (fx::match_head compares them instruction by instruction, whatever the slot numbering, the
// number of classes, rows and images and the threshold) can run as ONE launch of
// fx_head_stream instead of the two passes of the generic row compaction; every other region
// is untouched.  Results are bit-identical to the generic kernels: same device functions, same
// order of operations.
#pragma once
#include <stdint.h>

#include <algorithm>

#include "fx_bytecode.h"

#define FX_HEAD_SUB 256u       // most rows of a sub-tile (FX_BLOCK: one kept row a lane)
#define FX_HEAD_NSUB 4u        // ballots of a chunk: it holds at most FX_BLOCK rows
#define FX_HEAD_KV 6u          // 128-bit loads per lane that carry a sub-tile
#define FX_HEAD_STATUS_BITS 9u // a chunk's count is at most FX_BLOCK
#define FX_HEAD_MIN_CHUNK 64u  // fewest rows of a chunk unless the image has fewer
#define FX_HEAD_FULL_CHUNKS 384u   // chunks of FX_BLOCK rows from which on a launch has no smaller ones
#define FX_HEAD_ONE_A_CU 256u
// hash of the normalised programs of the detection-head region (fx_head_match.cpp)
#define FX_HEAD_NORM_HASH 0xed6ab9314c50ff65ull
// the same region with the anchors folded into box centres [N, 2] and half sizes [N, 2] and the
// strides as [N, 1] (what constant propagation leaves of anchors generated from static shapes)
#define FX_HEAD_NORM_HASH_FOLDED 0x680166c2c9e835ddull

// What the matcher found (host).
struct FxHeadInfo {
  bool ok = false;
  bool ragged = false;           // as ok, but rows of class scores that are no whole groups of four
  uint64_t norm_hash = 0;        // hash of the normalised programs (reported also when they do not match)
  uint32_t pred_slot = 0, anc_slot = 0, strd_slot = 0;   // pointer slots (FX_SLOT_TASK: per-task table)
  int32_t pred_tcoef = 0, anc_tcoef = 0, strd_tcoef = 0; // element offset per task
  bool folded = false;           // centres and half sizes instead of anchors: anc_* is the centres', half_* the half sizes'
  uint32_t half_slot = 0;
  int32_t half_tcoef = 0;
  uint32_t S = 0, C = 0;         // floats per prediction row (5 + C), classes
  uint32_t thr_bits = 0;         // objectness threshold (float bits)
  uint32_t n_rows = 0, n_tasks = 0;
  uint32_t out_slot[3] = {0, 0, 0};      // objectness [K], boxes [K, 4], class scores [K, C]
  uint32_t out_tstride[3] = {0, 0, 0};   // element offset per task
  uint32_t slot_total = 0;
};

// Kernel arguments (by value, followed by the FxDyn block in the argument segment).
struct FxHeadLaunch {
  uint32_t n_rows, n_tasks;
  uint32_t chunks, chunk_rows;   // workgroups per task and rows of each (<= FX_BLOCK)
  uint32_t sub_rows;             // rows of a sub-tile (<= FX_HEAD_SUB; the window holds them)
  uint32_t S, C;
  uint32_t g_magic, g_shift;     // fast division by C / 4 (groups of four class scores per row); C % 4 != 0: by C
  uint32_t thr_bits;
  uint32_t epoch, spin_limit;
  uint32_t n_sptr, n_tptr;
  uint32_t pred_slot, anc_slot, strd_slot;
  int32_t pred_tcoef, anc_tcoef, strd_tcoef;
  uint32_t out_slot[3], out_tstride[3];
  uint32_t bulk_delay;           // big launches: waves without a gather wait this long (units of 64 clocks) before they ask for rows
  uint32_t folded;               // 1: anc_slot holds box centres [N, 2], half_slot half sizes [N, 2]
  uint32_t half_slot;
  int32_t half_tcoef;
  uint32_t* status;              // one word per chunk, tagged with the epoch
  uint32_t* totals;              // pinned host memory: kept rows per task
};
static_assert(sizeof(FxHeadLaunch) % 8 == 0, "the FxDyn block follows at an 8-byte boundary");

// Rows that the loads of a sub-tile carry.
inline uint32_t fx_head_carried(uint32_t S) { return std::min<uint32_t>(FX_HEAD_SUB, (FX_HEAD_KV * FX_BLOCK * 4u - 6u) / S); }
inline uint32_t fx_head_window_bytes(uint32_t rows, uint32_t S) { return (((rows * S + 3u + 3u) >> 2) + 1u) * 16u; }

// Rows of a chunk and of a sub-tile.  slots(rows): workgroups that the device holds at once with a window of so
// many rows.  Every image's rows are dealt to its workgroups in equal runs, as few workgroups as give every slot
// one, but chunks have at least
//   256 rows where one round of loads carries them and that still makes FX_HEAD_FULL_CHUNKS (one and a half a CU),
//   192 where one round carries them, or in such a launch two do, 128 where two do, and 64:
// a workgroup looks back over the chunks of its image ahead of it, some 200 of them otherwise.  A launch that would have
// less than a workgroup for every CU takes no larger chunks than make 64 an image, which is one look.  Call, us, least rows
// 64 : 128 : 192 : 256: one image of 608, 8 classes 13.2 : 12.3 : 12.1 : 13.0; four of 320 13.1 : 12.5 : 12.7 : 13.3; nine of
// 480, 5 classes 20.4 : 17.7 : 17.1 : 16.2, 13 19.2 : 18.7 : 18.7 : 18.2; sixteen of 416, 5 22.4 : 22.8 : 22.5 : 20.9, 28
// 22.8 : 22.5 : 21.5 : 21.1; one of 416, 50 classes 12.9 : 12.7 : 14.4 : 14.8, 60 12.7 : 12.1 : 13.0 : 13.3; nine of 480, 75
// 20.8 : 20.6 : 22.9 : 25.8; one of 224, 90 11.1 : 11.8 : 15.4 : 19.5.
//   A chunk takes as few rounds as the loads allow, each a sub-tile, and the window holds the rows of one: LDS beyond
// that costs workgroups.  (Twelve of 608, 13 classes, one round of 153 rows instead of three: kernel 20.8 -> 11.7.)
// How long (units of 64 clocks) waves that gather no objectness hold their first rows back, so that the counts that
// later workgroups wait for are not in a queue behind them.  That pays by the bytes of a launch and by the rows that are to
// be counted; us, held back 0 : 64 : 128 units:
//   rows     MB
//   31 941   8.3  14.3 : 15.2 : 16.6      170 352   4.8  19.6 : 18.3 : 19.9      127 575  28.1  26.8 : 21.1 : 21.1
//   49 392   8.9  17.9 : 18.2 : 20.0      127 449   7.7  16.5 : 15.0 : 16.8      272 916  14.2  22.8 : 19.8 : 20.3
//   31 941  12.1  13.9 : 14.4 : 16.1      170 352  12.3  21.1 : 18.4 : 19.8      272 916  19.7  23.6 : 22.8 : 19.7
//   61 740   8.2  19.3 : 19.5 : 21.2      272 916   6.6  22.8 : 18.8 : 20.3      170 352  22.5  27.8 : 23.4 : 22.1
//   64 000  24.3  19.9 : 16.5 : 17.6      170 352  17.0  23.7 : 22.0 : 21.3      127 449  33.1  28.7 : 21.4 : 21.3
//   63 882   8.4  16.2 : 15.8 : 17.3      127 449  16.8  20.1 : 17.7 : 17.6      272 916  27.3  28.2 : 26.2 : 21.4
inline uint32_t fx_head_hold_back(uint32_t n_rows, uint32_t n_tasks, uint32_t S) {
  const double rows = (double)n_rows * n_tasks, bytes = rows * S * 4.0;
  return bytes >= 16e6 && rows >= 150e3 ? 128u : bytes * rows >= 5e11 ? 64u : 0u;
}

struct FxHeadGeometry { uint32_t chunk_rows, sub_rows; };
template <class Slots>
FxHeadGeometry fx_head_geometry(uint32_t n_rows, uint32_t n_tasks, uint32_t S, Slots&& slots) {
  const uint32_t rows = std::max<uint32_t>(n_rows, 1u), tasks = std::max<uint32_t>(n_tasks, 1u), carried = fx_head_carried(S);
  const uint64_t full = (uint64_t)tasks * ((rows + FX_BLOCK - 1u) / FX_BLOCK);
  const bool many = full >= FX_HEAD_FULL_CHUNKS;
  uint32_t least = many && carried >= FX_BLOCK ? FX_BLOCK : carried >= (many ? 96u : 192u) ? 192u : carried >= 64u ? 128u : FX_HEAD_MIN_CHUNK;
  if ((uint64_t)tasks * ((rows + least - 1u) / least) < FX_HEAD_ONE_A_CU) least = std::min(least, std::max<uint32_t>(FX_HEAD_MIN_CHUNK, (rows + 63u) / 64u));
  least = std::min(least, rows);
  auto chunk = [&](uint32_t window) {
    const uint32_t per_task = std::max<uint32_t>(1u, (uint32_t)slots(window) / tasks);
    return std::min<uint32_t>(FX_BLOCK, std::max<uint32_t>((rows + per_task - 1u) / per_task, least));
  };
  for (uint32_t window = std::min<uint32_t>(carried, 64u);;) {   // (a larger window: fewer slots, not fewer rows)
    const uint32_t cr = chunk(window), rounds = (cr + carried - 1u) / carried, sub = (cr + rounds - 1u) / rounds;
    if (sub <= window) return FxHeadGeometry{cr, sub};
    window = sub;
  }
}
