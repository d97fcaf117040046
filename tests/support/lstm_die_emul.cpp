// TEST INFRASTRUCTURE ONLY - never linked into or loaded by the product.
//
// CPU build of the schedule and hand-over of fx_lstm_die_kernel (fx_lstm_sched.h: a sequence on one die): one
// host thread per workgroup, stages of layers whose steps are their own, the two parities of the h buffer, the
// ring between stages with its counts of read vectors, tags from launch to launch.
#include <math.h>
#include <string.h>

#include <functional>
#include <thread>
#include <vector>

#include "../../functs_amd/csrc/fxhip/fx_lstm_groups.h"
#include "../../functs_amd/csrc/fxhip/fx_lstm_sched.h"

namespace {
struct HostAtomics {
  static uint32_t add(uint32_t* p) { return __atomic_fetch_add(p, 1u, __ATOMIC_ACQ_REL); }
  static uint32_t load(uint32_t* p) { return __atomic_load_n(p, __ATOMIC_ACQUIRE); }
  static void store(uint32_t* p, uint32_t v) { __atomic_store_n(p, v, __ATOMIC_RELEASE); }
  static void store64(uint64_t* p, uint64_t v) { __atomic_store_n(p, v, __ATOMIC_RELEASE); }
};
float sigmoidf(float x) { return 1.0f / (1.0f + expf(-x)); }

// n_wg workgroups a stage (at most FX_LSTM_DIE_WG), H / n_wg units each; slow: (stage, workgroup) that dawdles, stop: that
// leaves after four steps
struct Run {
  FxLstmArgs a;
  int L, n_wg, total, slow_stage, slow_wg, stop_stage = -1, stop_wg = -1;
  bool give_up(uint32_t polls) const {
    if (polls <= a.spin_limit && !((polls & 255u) == 0u && HostAtomics::load(a.ctl + FX_LSTM_W_ERR) != 0u)) return false;
    HostAtomics::store(a.ctl + FX_LSTM_W_ERR, 1u);
    return true;
  }
  template <class F>
  bool wait(F&& there) const {
    for (uint32_t polls = 0; !there();) {
      if (give_up(++polls)) return false;
      std::this_thread::yield();
    }
    return true;
  }
  void workgroup(int b, int stage, int gi) const {
    const bool refused = fx_lstm_refused<HostAtomics>(a);
    const bool done = !refused && steps(b, stage, gi);
    if (refused) *a.err_host = 2u;
    if (!done && !(stage == stop_stage && gi == stop_wg)) fx_lstm_poison(a, L, 0u, 1u);
  }
  bool steps(int b, int stage, int gi) const {
    const int H = a.H, B = a.B, T = a.T, NL = fx_lstm_stage_layers(H, L), stages = L / NL, U = H / n_wg, u0 = gi * U, j0 = stage * NL;
    const uint32_t base = HostAtomics::load(a.ctl + FX_LSTM_W_BASE);
    const FxLstmDieArea area = fx_lstm_die_area(B, H, L);
    const int n_steps = fx_lstm_stage_steps(T, NL);
    uint64_t* ring_in = a.hbuf + area.ring + (size_t)((stage - 1) * B + b) * (FX_LSTM_RING * H);
    uint64_t* ring_out = a.hbuf + area.ring + (size_t)(stage * B + b) * (FX_LSTM_RING * H);
    uint64_t* read_in = a.hbuf + area.read + ((stage - 1) * B + b) * FX_LSTM_DIE_WG + gi;
    uint64_t* read_out = a.hbuf + area.read + (stage * B + b) * FX_LSTM_DIE_WG;
    std::vector<std::vector<float>> in(3, std::vector<float>(H)), below(NL, std::vector<float>(H)), hv(NL, std::vector<float>(H));
    std::vector<float> c((size_t)NL * U);
    for (int k = 0; k < NL; ++k)
      for (int u = 0; u < U; ++u) c[k * U + u] = a.c0 ? a.c0[((size_t)(j0 + k) * B + b) * H + u0 + u] : 0.0f;
    // element i of the vector p, once it carries `tag`
    auto tagged = [&](uint64_t* p, uint32_t tag, float* to) {
      return wait([&] {
        const uint64_t e = __atomic_load_n(p, __ATOMIC_ACQUIRE);
        const uint32_t bits = (uint32_t)e;
        memcpy(to, &bits, 4);
        return fx_lstm_tag_of(e) == tag;
      });
    };
    auto park = [&](int t) {
      if (t >= T) return true;
      for (int i = 0; i < H; ++i) {
        if (stage == 0) in[t % 3][i] = a.x[((size_t)t * B + b) * H + i];
        else if (!tagged(ring_in + (size_t)(t % FX_LSTM_RING) * H + i, base + (uint32_t)t + 1u, &in[t % 3][i])) return false;
      }
      if (stage > 0) HostAtomics::store64(read_in, (uint64_t)(base + (uint32_t)t + 1u));
      return true;
    };
    if (!park(0) || !park(1)) return false;
    for (int d = 0; d < n_steps; ++d) {
      if (stage == stop_stage && gi == stop_wg && d == 4) return false;
      if (stage == slow_stage && gi == slow_wg && d % 5 == 0) std::this_thread::sleep_for(std::chrono::milliseconds(2));
      for (int k = 0; k < NL; ++k) {
        const int t = fx_lstm_stage_time(d, k, T);
        const bool need = d > 0 && fx_lstm_stage_time(d - 1, k, T) >= 0 && (t >= 0 || k + 1 < NL);
        for (int i = 0; i < H; ++i) {
          hv[k][i] = t == 0 && a.h0 ? a.h0[((size_t)(j0 + k) * B + b) * H + i] : 0.0f;
          if (need && !tagged(a.hbuf + fx_lstm_hoff((d + 1) & 1, j0 + k, b, i, L, B, H), fx_lstm_tag_read(base, d), &hv[k][i])) return false;
        }
      }
      for (int k = 0; k < NL; ++k) {
        const int t = fx_lstm_stage_time(d, k, T), j = j0 + k;
        if (t < 0) continue;
        const std::vector<float>& x = k == 0 ? in[d % 3] : below[k - 1];
        for (int u = 0; u < U; ++u) {
          float g[4];
          for (int q = 0; q < 4; ++q) {
            float s = 0.f;
            for (int i = 0; i < H; ++i) {
              const size_t w = ((size_t)(j * 4 + q) * H + i) * H + u0 + u;
              s += a.wih[w] * x[i] + a.whh[w] * hv[k][i];
            }
            g[q] = s + a.bih[(size_t)(j * 4 + q) * H + u0 + u] + a.bhh[(size_t)(j * 4 + q) * H + u0 + u];
          }
          float& cell = c[k * U + u];
          cell = sigmoidf(g[1]) * cell + sigmoidf(g[0]) * tanhf(g[2]);
          const float h = sigmoidf(g[3]) * tanhf(cell);
          uint32_t bits;
          memcpy(&bits, &h, 4);
          HostAtomics::store64(a.hbuf + fx_lstm_hoff(d & 1, j, b, u0 + u, L, B, H), fx_lstm_pack(bits, fx_lstm_tag_written(base, d)));
          if (k == NL - 1 && stage + 1 < stages) HostAtomics::store64(ring_out + (size_t)(t % FX_LSTM_RING) * H + u0 + u, fx_lstm_pack(bits, base + (uint32_t)t + 1u));
          if (j == L - 1) a.out[((size_t)t * B + b) * H + u0 + u] = h;
          if (t == T - 1) {
            a.state_h[((size_t)j * B + b) * H + u0 + u] = h;
            a.state_c[((size_t)j * B + b) * H + u0 + u] = cell;
          }
        }
      }
      below = hv;
      if (!park(d + 2)) return false;
      if (stage + 1 < stages && d + 1 < n_steps && d % (FX_LSTM_RING / 2) == FX_LSTM_RING / 2 - 1) {
        const int seen = d + 1 - FX_LSTM_RING / 2;
        for (int w = 0; w < n_wg && seen > 0; ++w)
          if (!wait([&] { return (int32_t)((uint32_t)__atomic_load_n(read_out + w, __ATOMIC_ACQUIRE) - (base + (uint32_t)seen)) >= 0; })) return false;
      }
    }
    fx_lstm_leave<HostAtomics>(a.ctl, (uint32_t)total, base, (uint32_t)n_steps + 1u, a.hbuf, area.words);
    return true;
  }
};
}  // namespace

// `launches` runs on one workspace that is cleared once; the error word, or -1 when the workspace was not left
// as the next launch needs it
extern "C" int fx_lstm_die_emul(const float* x, const float* wih, const float* whh, const float* bih, const float* bhh, const float* h0,
                                const float* c0, float* out, float* state_h, float* state_c, int T, int B, int H, int L, int n_wg,
                                uint32_t spin_limit, int launches, uint32_t base0, int slow_stage, int slow_wg) {
  if (!fx_lstm_die_fits(B, H, L)) return -2;
  std::vector<uint32_t> ctl(FX_LSTM_CTL_WORDS, 0u);
  std::vector<uint64_t> area(fx_lstm_die_area(B, H, L).words, 0ull);
  ctl[FX_LSTM_W_BASE] = base0;
  Run r;
  r.a = FxLstmArgs{x, wih, whh, bih, bhh, h0, c0, out, state_h, state_c, area.data(), ctl.data(), ctl.data(), ctl.data(), nullptr, T, B, H, spin_limit};
  const int stages = L / fx_lstm_stage_layers(H, L);
  r.L = L; r.n_wg = n_wg; r.total = stages * B * n_wg; r.slow_stage = slow_stage; r.slow_wg = slow_wg;
  uint32_t base = base0;
  for (int n = 0; n < launches; ++n) {
    for (size_t i = 0; i < (size_t)T * B * H; ++i) out[i] = NAN;
    std::vector<std::thread> th;
    for (int b = 0; b < B; ++b)
      for (int s = 0; s < stages; ++s)
        for (int g = 0; g < n_wg; ++g) th.emplace_back(&Run::workgroup, std::cref(r), b, s, g);
    for (auto& t : th) t.join();
    if (ctl[FX_LSTM_W_ERR]) return (int)ctl[FX_LSTM_W_ERR];
    base += (uint32_t)fx_lstm_stage_steps(T, fx_lstm_stage_layers(H, L)) + 1u;
    if (base >= FX_LSTM_TAG_WRAP) {
      base = 0u;
      for (uint64_t e : area)
        if (e != 0ull) return -1;
    }
    if (ctl[FX_LSTM_W_BASE] != base || ctl[FX_LSTM_W_LEAVE] != 0u) return -1;
  }
  return 0;
}

// A workgroup (stop_stage, stop_wg) leaves in the middle; then, with whatever that left, another launch; then, on a
// cleared workspace, one with the error word of control area `marked` set (0: its own, 1, 2: the other forms'); then one with
// all clear.  Bits: 1 the first gave up; 2 with NaN for results; 4 the second was refused; 8 with NaN; 16 the marked one
// was refused, 32 with NaN; 64 the last one ran.
extern "C" int fx_lstm_die_emul_give_up(const float* x, const float* wih, const float* whh, const float* bih, const float* bhh, const float* h0,
                                        const float* c0, float* out, float* state_h, float* state_c, int T, int B, int H, int L, int n_wg,
                                        uint32_t spin_limit, int stop_stage, int stop_wg, int marked) {
  std::vector<uint32_t> ctl[3];
  for (auto& c : ctl) c.assign(FX_LSTM_CTL_WORDS, 0u);
  std::vector<uint64_t> area(fx_lstm_die_area(B, H, L).words, 0ull);
  uint32_t err = 0u;
  Run r;
  r.a = FxLstmArgs{x, wih, whh, bih, bhh, h0, c0, out, state_h, state_c, area.data(), ctl[0].data(), ctl[1].data(), ctl[2].data(), &err, T, B, H, spin_limit};
  const int stages = L / fx_lstm_stage_layers(H, L);
  r.L = L; r.n_wg = n_wg; r.total = stages * B * n_wg; r.slow_stage = r.slow_wg = -1;
  auto launch = [&] {
    err = 0u;
    for (size_t i = 0; i < (size_t)T * B * H; ++i) out[i] = 1.0f;
    std::vector<std::thread> th;
    for (int b = 0; b < B; ++b)
      for (int s = 0; s < stages; ++s)
        for (int g = 0; g < n_wg; ++g) th.emplace_back(&Run::workgroup, std::cref(r), b, s, g);
    for (auto& t : th) t.join();
  };
  // (the workgroup that left in the middle, or others ahead of it, may have written steps of theirs behind the NaNs: the last step
  // nobody has reached)
  auto all_nan = [&] {
    for (int i = 0; i < B * H; ++i)
      if (!isnan(out[(size_t)(T - 1) * B * H + i])) return false;
    return true;
  };
  int bits = 0;
  r.stop_stage = stop_stage; r.stop_wg = stop_wg;
  launch();
  bits |= (ctl[0][FX_LSTM_W_ERR] ? 1 : 0) | (all_nan() ? 2 : 0);
  r.stop_stage = r.stop_wg = -1;
  launch();
  bits |= (err == 2u ? 4 : 0) | (all_nan() ? 8 : 0);
  for (auto& c : ctl) c.assign(FX_LSTM_CTL_WORDS, 0u);
  area.assign(area.size(), 0ull);
  r.a.ctl = ctl[0].data(); r.a.ctl_other = ctl[1].data(); r.a.ctl_third = ctl[2].data(); r.a.hbuf = area.data();
  ctl[marked][FX_LSTM_W_ERR] = 1u;
  launch();
  bits |= (err == 2u ? 16 : 0) | (all_nan() ? 32 : 0);
  ctl[marked][FX_LSTM_W_ERR] = 0u;
  r.a.spin_limit = 1u << 30;
  launch();
  return bits | (err == 0u && ctl[0][FX_LSTM_W_ERR] == 0u ? 64 : 0);
}

// Streams 0 .. n - 1 launch once each, in that order, then stream 0 `more` times, in groups that hold `device`: have
// others than `stream` launched lately?
extern "C" int fx_lstm_others_emul(int n, int more, uint32_t need, uint32_t device, int stream) {
  FxLstmGroups g;
  bool joins;
  for (int s = 0; s < n + more; ++s) g.admit(s < n ? (uint64_t)s : 0u, 0u, need, device, true, &joins).last = ++g.launches;
  return g.others((uint64_t)stream, 0u) ? 1 : 0;
}
