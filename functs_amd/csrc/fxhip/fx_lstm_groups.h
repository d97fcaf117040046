// Which launches of the persistent LSTM kernels may be on a device at the same time.  A workgroup of such
// a kernel waits for values of all the others, so a launch ends only if all its workgroups get a place:
// two launches that are half resident each wait for ever (until their bounded waits are given up).  The
// text builds for the CPU as well, where a test runs it (tests/support/lstm_emul.cpp).
//
// A launch needs grid / r compute units, r = how many of its workgroups fit one, rounded down to a power
// of two (unit: FX_LSTM_CU-ths).  r counts every workgroup as a whole number of waves for each of the
// compute unit's four SIMDs (fx_lstm_block): which SIMD gets the odd waves is the hardware's choice, and two
// workgroups of ten waves of 96 registers, which would fit with five waves on each, do not with six on one.
// Launches whose needs together are at most the device all get their
// places, whatever the order in which the workgroups arrive: take the smallest of those that still have
// workgroups without a place (smaller ones end by themselves).  If no compute unit had room for one more,
// every one would be full, for what the others take of it is a multiple of what this one takes; but one
// workgroup is not there yet, so less than the device is taken.
// Launches come in groups that fit together, and a group starts when the one before it has ended: a
// stream's first launch of a group waits for the last launches of the group before (events, on the
// device).  A program with one stream never waits; on four streams four stacks of 512 units, two layers, one sequence
// each, run at the same time, and two that take the whole device run one after the other.
// Events: the legacy default stream always exists and is never captured, so its event is recorded when a group
// closes, from whichever thread that is, and launches on it cost nothing.  On any other stream an event is
// recorded behind every launch: when it is wanted the stream may be gone, or capturing.
#pragma once
#include <stdint.h>

#include <initializer_list>
#include <vector>

#define FX_LSTM_CU 64u

inline uint32_t fx_lstm_block(uint32_t threads) { return (threads + 255u) & ~255u; }
inline uint32_t fx_lstm_need(uint32_t grid, uint32_t per_cu) {
  uint32_t r = 1u;
  while (2u * r <= per_cu && 2u * r <= FX_LSTM_CU) r *= 2u;
  return grid * (FX_LSTM_CU / r);
}

struct FxLstmGroups {
  struct Member {
    uint64_t stream, thread;   // (thread: for the streams that every thread has of its own)
    uint32_t need;             // the largest of the stream's launches in the group: one of them runs at a time
    void* done;                // event behind the last of them (null: none was made yet)
    bool late;                 // ... which is recorded when the group has closed (close_late), not behind every launch
    uint64_t last = 0;         // number of its last launch
  };
  std::vector<Member> now, before;
  uint64_t launches = 0;
  std::vector<void*> spare;    // events to use again

  static bool same(const Member& m, uint64_t stream, uint64_t thread) { return m.stream == stream && m.thread == thread; }
  // The member that a launch belongs to.  *joins: its stream has to wait for the others' events of the group
  // before (wait) ahead of it, once close_late has recorded the late ones.
  Member& admit(uint64_t stream, uint64_t thread, uint32_t need, uint32_t device, bool late, bool* joins) {
    uint64_t total = need;
    Member* mine = nullptr;
    for (Member& m : now) {
      if (same(m, stream, thread)) mine = &m;
      total += same(m, stream, thread) ? (m.need > need ? m.need - need : 0u) : m.need;
    }
    if (total > device && !(mine && now.size() == 1)) {   // (alone there is nobody to wait for)
      for (const Member& m : before)
        if (m.done) spare.push_back(m.done);
      before.swap(now);
      now.clear();
      mine = nullptr;
    }
    *joins = !mine;
    if (mine) {
      if (mine->need < need) mine->need = need;
      return *mine;
    }
    now.push_back(Member{stream, thread, need, nullptr, late});
    return now.back();
  }
  // Whether other streams than this one have launched lately: a form that holds every die would make the streams
  // take turns.  (Counted in launches and not asked of the device: queries are not allowed
  // beside a capture.)
  bool others(uint64_t stream, uint64_t thread) const {
    for (const std::vector<Member>* group : {&now, &before})
      for (const Member& m : *group)
        if (!same(m, stream, thread) && launches - m.last < 64u) return true;
    return false;
  }
  void* event_to_use() {
    if (spare.empty()) return nullptr;
    void* e = spare.back();
    spare.pop_back();
    return e;
  }
  // record(Member&): gives the member its event and records it on its stream; false: it could not
  template <class F>
  bool close_late(F&& record) {
    for (Member& m : before)
      if (m.late) {
        if (!record(m)) return false;
        m.late = false;
      }
    return true;
  }
  template <class F>
  bool wait(uint64_t stream, uint64_t thread, F&& wait_for) {
    for (const Member& m : before)
      if (m.done && !same(m, stream, thread) && !wait_for(m.done)) return false;   // (no event: its launch failed)
    return true;
  }
  // the launch that joined last did not get as far as that
  void withdraw() {
    if (now.back().done) spare.push_back(now.back().done);
    now.pop_back();
  }
};
