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
// device).  A program with one stream never waits; on two streams two stacks of 512 units, one sequence
// each, run at the same time, and two that take the whole device run one after the other.
#pragma once
#include <stdint.h>

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
    void* done;                // event behind the last of them
  };
  std::vector<Member> now, before;
  std::vector<void*> spare;    // events to use again

  // The member that a launch belongs to.  wait_for: events that its stream has to wait for ahead of it.
  // `done` is null for a new member that got no spare event.
  Member& admit(uint64_t stream, uint64_t thread, uint32_t need, uint32_t device, std::vector<void*>* wait_for) {
    wait_for->clear();
    auto same = [&](const Member& m) { return m.stream == stream && m.thread == thread; };
    uint64_t total = need;
    Member* mine = nullptr;
    for (Member& m : now) {
      if (same(m)) mine = &m;
      total += same(m) ? (m.need > need ? m.need - need : 0u) : m.need;
    }
    if (total > device && !(mine && now.size() == 1)) {   // (alone there is nobody to wait for)
      for (const Member& m : before) spare.push_back(m.done);
      before.swap(now);
      now.clear();
      mine = nullptr;
    }
    if (mine) {
      if (mine->need < need) mine->need = need;
      return *mine;
    }
    for (const Member& m : before)
      if (!same(m)) wait_for->push_back(m.done);
    now.push_back(Member{stream, thread, need, nullptr});
    if (!spare.empty()) {
      now.back().done = spare.back();
      spare.pop_back();
    }
    return now.back();
  }
};
