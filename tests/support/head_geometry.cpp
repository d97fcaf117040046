// TEST INFRASTRUCTURE ONLY - never linked into or loaded by the product.
//
// fx_head_geometry on a model of the device: 256 compute units of eight workgroups and 160 KB of LDS each.
#include "../../functs_amd/csrc/fxhip/fx_head.h"

extern "C" void fx_head_geometry_of(uint32_t n_rows, uint32_t n_tasks, uint32_t S, uint32_t* out) {
  const FxHeadGeometry g = fx_head_geometry(n_rows, n_tasks, S, [&](uint32_t window) {
    const uint32_t per_cu = std::min<uint32_t>(8u, (160u << 10) / (fx_head_window_bytes(window, S) + 1400u));
    return 256u * (per_cu >= 3u ? per_cu - 1u : per_cu);
  });
  out[0] = g.chunk_rows;
  out[1] = g.sub_rows;
  out[2] = fx_head_carried(S);
  out[3] = fx_head_window_bytes(g.sub_rows, S);
}
