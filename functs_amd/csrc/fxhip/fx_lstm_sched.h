// Schedule and hand-over protocol of the persistent stacked-LSTM kernel (fx_lstm.hip), written so
// that the same text also builds for the CPU, where tests run it with one host thread per
// workgroup (tests/support/lstm_emul.cpp) to check the schedule, the buffer parities and the
// protocol without a GPU.
//
// The recurrence (functs/benchmark/ai_model/lstm/lstm.py:79-133): for t in [0, T), for layer j in
// [0, L): gates(t, j) need the output of layer j - 1 at time t and the state of layer j at time
// t - 1.  Cells (t, j) with the same d = t + j are independent, so the kernel walks the
// T + L - 1 diagonals d and computes every active layer of a diagonal in one step.
//   h of (t, j), computed in step d, is written to hbuf[d & 1][j]; step d reads its inputs from
//   hbuf[(d - 1) & 1] (layer j - 1 at time t and layer j at time t - 1 were both computed in
//   step d - 1), from x (layer 0) and from h0 (t == 0).
// Hand-over without a barrier: every element of hbuf is 64 bits, the value and the TAG of the
// step that wrote it (one atomic store), and a reader polls the elements it needs until they
// carry the tag of the step it expects.  A workgroup writes step d only after it has read all
// it needs of step d - 1, and nobody can be in step d + 1, whose writes land on the parity that
// step d reads, before every workgroup has written step d: the two parities suffice.
// Tags are base + d + 1, where base is a word of the workspace that the last workgroup to leave
// advances past the tags of the launch, so the elements a launch finds from earlier launches
// never carry a tag it waits for (a zeroed workspace carries tag 0, which no step has).
// Every poll loop is bounded: a reader that gives up sets the error word and its workgroup
// leaves; the others give up in turn.
#pragma once
#include <stdint.h>

#ifndef FX_LSTM_HD
#define FX_LSTM_HD
#endif

#define FX_LSTM_LINE 64u                          // words between the control words: one 256-byte line each
#define FX_LSTM_W_BASE 0u                         // tag base of the next launch
#define FX_LSTM_W_LEAVE (1u * FX_LSTM_LINE)       // workgroups that have left
#define FX_LSTM_W_ERR (2u * FX_LSTM_LINE)         // a wait was given up
#define FX_LSTM_CTL_WORDS (3u * FX_LSTM_LINE)
#define FX_LSTM_TAG_WRAP 0x80000000u              // the base starts over (and the tags are cleared, fx_lstm_leave) beyond this

// The second hand-over, of the kernel for groups of rows (one row at a time goes by tags): an element is ONE
// 32-bit word, its value with all bits inverted, and 0 says that it has not been written yet (the
// word that would be 0, a NaN of all ones, is written as another NaN).  Half the bytes of a value with
// its tag, and what all workgroups read in a step is what a step waits for.
//   Four slots of [L][B][H] words, used in turn: step d writes slot (base + d) & 3, reads slot
//   (base + d - 1) & 3, and its owners clear their words of slot (base + d + 2) & 3.
//   Clearing is safe: behind the barrier of step d a workgroup has seen every value of step d - 1, so
//   every workgroup is past its reads of step d - 1, which were reads of slot d - 2, the one cleared.
//   A cleared word is seen in time: a workgroup lets its clears of step d be acknowledged before its
//   barrier of step d + 1, ahead of its values of step d + 1; who reads slot d + 2 (in step d + 3) has
//   seen those values.
//   base is a word of the workspace, advanced by the steps of every launch: slots base and base + 1 are
//   clear when a launch begins (all four in a zeroed workspace), and stay so from launch to launch.
FX_LSTM_HD inline uint32_t fx_lstm_slot(uint32_t base, int d) { return (base + (uint32_t)d) & 3u; }
FX_LSTM_HD inline uint32_t fx_lstm_word(uint32_t value_bits) { return value_bits == 0xffffffffu ? ~0x7fc00000u : ~value_bits; }
FX_LSTM_HD inline uint32_t fx_lstm_word_value(uint32_t word) { return ~word; }

// arguments of the kernel (contiguous fp32 tensors; see fx_lstm_stack in include/fxhip.h)
struct FxLstmArgs {
  const float *x, *wih, *whh, *bih, *bhh;
  const float *h0, *c0;   // null: zero initial state
  float *out, *state_h, *state_c;
  uint64_t* hbuf;      // [2][L][B][H] (value, tag): h of the cells of the last two steps
  uint32_t* ctl;       // FX_LSTM_CTL_WORDS control words
  uint32_t* ctl_other; // those of the other hand-over: a wait that was given up in either refuses both
  uint32_t* ctl_third; // and those of the third one (its own again where there is none)
  uint32_t* err_host;  // pinned word that a given-up wait reports to as well (may be null)
  int T, B, H;
  uint32_t spin_limit;
};

FX_LSTM_HD inline int fx_lstm_steps(int T, int L) { return T > 0 ? T + L - 1 : 0; }
FX_LSTM_HD inline int fx_lstm_time(int d, int j, int T) {
  const int t = d - j;
  return (t >= 0 && t < T) ? t : -1;
}
// element offset of h of (layer j, batch b, unit u) in parity p of hbuf[2][L][B][H]
FX_LSTM_HD inline uint32_t fx_lstm_hoff(int p, int j, int b, int u, int L, int B, int H) {
  return (uint32_t)((((p * L + j) * B + b) * H) + u);
}
FX_LSTM_HD inline uint64_t fx_lstm_pack(uint32_t value_bits, uint32_t tag) { return ((uint64_t)tag << 32) | value_bits; }
FX_LSTM_HD inline uint32_t fx_lstm_tag_of(uint64_t e) { return (uint32_t)(e >> 32); }
// tag of what step d writes / of what step d reads (written by step d - 1)
FX_LSTM_HD inline uint32_t fx_lstm_tag_written(uint32_t base, int d) { return base + (uint32_t)d + 1u; }
FX_LSTM_HD inline uint32_t fx_lstm_tag_read(uint32_t base, int d) { return base + (uint32_t)d; }

// A wait that was given up: the launch's results are not to be used, and its workspace stays
// marked (the error word) until the host clears it.  Two rules make that visible in the data
// itself, whatever the caller does with the error report:
//   a workgroup that gives up fills out, state_h and state_c with NaN before it leaves (a
//   workgroup that has already finished may write a few values after that; the report still says
//   that the launch failed);
//   a launch that finds the error word set does no step at all: every workgroup reports the
//   error again, fills the results with NaN and leaves.
template <class A>
FX_LSTM_HD inline bool fx_lstm_refused(uint32_t* ctl) { return A::load(ctl + FX_LSTM_W_ERR) != 0u; }
// ... in any of its areas.  (The words are asked for together: one after the other they held up every launch's start, a batch of
// eight over eight steps 13.3 -> 13.7 us with the third.)
template <class A>
FX_LSTM_HD inline bool fx_lstm_refused(const FxLstmArgs& a) {
  const uint32_t e0 = A::load(a.ctl + FX_LSTM_W_ERR), e1 = A::load(a.ctl_other + FX_LSTM_W_ERR), e2 = A::load(a.ctl_third + FX_LSTM_W_ERR);
  return (e0 | e1 | e2) != 0u;
}
// element first, first + stride, ... of the three results
FX_LSTM_HD inline void fx_lstm_poison(const FxLstmArgs& a, int L, uint32_t first, uint32_t stride) {
  const float nan = __builtin_nanf("");
  const uint32_t n_out = (uint32_t)a.T * (uint32_t)a.B * (uint32_t)a.H, n_state = (uint32_t)L * (uint32_t)a.B * (uint32_t)a.H;
  for (uint32_t i = first; i < n_out; i += stride) a.out[i] = nan;
  for (uint32_t i = first; i < n_state; i += stride) {
    a.state_h[i] = nan;
    a.state_c[i] = nan;
  }
}

// A workgroup that has finished its last step checks out; the last one to do so (nobody reads
// or writes hbuf any more) moves the tag base past this launch's tags and puts the counter back
// to zero, so the same workspace serves the next launch on the stream without a clear in
// between.  Past FX_LSTM_TAG_WRAP the base starts over at zero, and the tags in hbuf are cleared
// first: at the memory side.  What the kernel on dies has stored to a die's cache only may be written
// back on top of that when the launch ends, and is overwritten by the next launch that waits for that
// place: a tag left over would have to lie untouched for 2^31 steps to be one that is waited for.
// A workgroup that gave up a wait does not check out: the error word stays set and the host clears the
// whole workspace before it is used again.
//   A: atomics policy { add(uint32_t*) -> old value, load(uint32_t*), store(uint32_t*, v), store64(uint64_t*, v) }
template <class A>
FX_LSTM_HD inline void fx_lstm_leave(uint32_t* ctl, uint32_t n_wg, uint32_t base, uint32_t n_steps, uint64_t* hbuf,
                                     uint32_t n_elems) {
  if (A::add(ctl + FX_LSTM_W_LEAVE) + 1u != n_wg) return;
  uint32_t next = base + n_steps;
  if (next >= FX_LSTM_TAG_WRAP) {
    for (uint32_t i = 0; i < n_elems; ++i) A::store64(hbuf + i, 0ull);
    next = 0u;
  }
  A::store(ctl + FX_LSTM_W_BASE, next);
  A::store(ctl + FX_LSTM_W_LEAVE, 0u);
}

// The same for the hand-over through words: the slots are as the next launch expects them.
template <class A>
FX_LSTM_HD inline void fx_lstm_leave_slots(uint32_t* ctl, uint32_t n_wg, uint32_t base, uint32_t n_steps) {
  if (A::add(ctl + FX_LSTM_W_LEAVE) + 1u != n_wg) return;
  A::store(ctl + FX_LSTM_W_BASE, (base + n_steps) & 3u);
  A::store(ctl + FX_LSTM_W_LEAVE, 0u);
}

// The third hand-over, of the kernel that keeps a sequence on one die (fx_lstm_die_kernel): its layers, or as
// many of them as the die's registers hold (a STAGE), run on the compute units that share a cache.
//   Steps of a stage are its own: in step d its layer k computes t = d - 2 k, so that what a layer needs of
//   the layer below was written two steps ago, and was read in the step before as that layer's own state.
//   The h of (stage's layer, t) travels as above, with its tag, through hbuf[d & 1][j]; the two parities suffice
//   for the same reason.
//   From stage to stage h travels through a ring of FX_LSTM_RING vectors with tags base + t + 1.  A stage runs
//   ahead of the next one, and overwrites vector t - FX_LSTM_RING of the ring only when all workgroups of the
//   next stage have published that they have read it (counts: base + vectors read).
#define FX_LSTM_RING 16
#define FX_LSTM_DIES 8        // dies of the chip, and
#define FX_LSTM_DIE_WG 32     // workgroups on each, one per compute unit
FX_LSTM_HD inline int fx_lstm_stage_steps(int T, int n_layers) { return T > 0 ? T + 2 * (n_layers - 1) : 0; }
FX_LSTM_HD inline int fx_lstm_stage_time(int d, int k, int T) {
  const int t = d - 2 * k;
  return (t >= 0 && t < T) ? t : -1;
}
// layers of a stage: all of them up to 256 units (their weights are at most 96 registers a lane), one of 512
FX_LSTM_HD inline int fx_lstm_stage_layers(int H, int L) { return H > 256 ? 1 : H == 256 && L == 4 ? 2 : L; }
FX_LSTM_HD inline bool fx_lstm_die_fits(int B, int H, int L) {
  return (H == 64 || H == 128 || H == 256 || H == 512) && L >= 1 && L <= 4 && B >= 1 && B * (L / fx_lstm_stage_layers(H, L)) <= FX_LSTM_DIES;
}
// A launch's start costs more on dies (one die fetches a layer's weights) and a step less, so the shortest sequences are the other
// forms', in calls and in captures.  The fewest steps that the kernel is taken for; speed of the best other form = 1, one step ahead of
// the line and at it (weights in the caches; from further away the kernel is ahead sooner): 64 units, three layers, eight sequences
// 0.94, 0.99, two layers, four 0.92, 1.06, one, one 0.89, 1.08; 128, four layers, four 1.00, 1.04; 256, three, four 0.97, 1.01; 512, one,
// eight 0.89, 0.96.  (Spread over the chip, 64 and 128 units lose up to a fifth between this line and some 16 steps: what is captured
// there has the bits of the calls instead.)
FX_LSTM_HD inline int fx_lstm_die_from(int B, int H, int L) {
  if (H <= 128 && B == 1) return 2;
  if (H == 64) return (L > 2 ? 5 : 3) + (B > 3) + (B > 5);
  if (H == 128) return L > 2 ? 5 : 3 + (B > 5);
  if (H == 256) return L == 4 ? 1 : L == 3 ? 5 : L + 1;
  return L == 1 && B > 4 ? 5 : L == 2 && B > 2 ? 3 : 1;
}
// The fewest steps for which its workgroups are placed on dies while nothing else is about; below, spread.  512 units, call
// on dies : spread : row by row, one sequence, one layer: 8 steps 23.0 : 18.6 : 21.6, 24 steps 40.3 : 40.1, 32 steps 49.0 : 50.9; two
// layers: 8 steps 27.7 : 27.4 : 30.0, 12 steps 32.1 : 33.0; two sequences: 16 steps 39.6 : 37.9, 24 steps 48.8 : 49.5; three
// layers: 8 steps 32.0 : 31.7, 12 steps 37.0 : 37.3.
FX_LSTM_HD inline int fx_lstm_die_alone(int B, int H, int L) { return H < 512 || L * B > 4 || L > 3 ? 1 : L == 1 ? 24 : L == 2 ? 10 * B : 10; }
// 64-bit words behind the control words: h [2][L][B][H]; rings [stages - 1][B][FX_LSTM_RING][H]; counts of read
// vectors [stages - 1][B][FX_LSTM_DIE_WG]; the die that every workgroup runs on [FX_LSTM_DIES][FX_LSTM_DIE_WG]
struct FxLstmDieArea { uint32_t ring, read, where, words; };
FX_LSTM_HD inline FxLstmDieArea fx_lstm_die_area(int B, int H, int L) {
  const uint32_t links = (uint32_t)(L / fx_lstm_stage_layers(H, L) - 1) * (uint32_t)B;
  FxLstmDieArea a;
  a.ring = (uint32_t)(2 * L * B * H);
  a.read = a.ring + links * (uint32_t)(FX_LSTM_RING * H);
  a.where = a.read + links * FX_LSTM_DIE_WG;
  a.words = a.where + FX_LSTM_DIES * FX_LSTM_DIE_WG;
  return a;
}
