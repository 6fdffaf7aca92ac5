// g2b_wide.hip - dispatch of k_wide (g2b_wide.h) over KV formats and head
// sizes; the kernels are compiled by g2b_wide_inst.hip.
#include "g2b_internal.h"

namespace g2b {

bool wide_available(const ShapeDev &sh) {
  if (sh.head_dim != 64 && sh.head_dim != 128 && sh.head_dim != 256) return false;
  if (sh.n_kv_heads <= 0 || sh.n_heads % sh.n_kv_heads) return false;
  return sh.n_heads / sh.n_kv_heads <= 16;
}

hipError_t launch_wide(const DecodeParams &p, int n_layers, hipStream_t s) {
  if (!wide_available(p.sh)) return hipErrorInvalidValue;
  if (p.sh.kv_q8) {
    switch (p.sh.head_dim) {
      case 64: return launch_wide_hd<1, 64>(p, n_layers, s);
      case 128: return launch_wide_hd<1, 128>(p, n_layers, s);
      default: return launch_wide_hd<1, 256>(p, n_layers, s);
    }
  }
  switch (p.sh.head_dim) {
    case 64: return launch_wide_hd<0, 64>(p, n_layers, s);
    case 128: return launch_wide_hd<0, 128>(p, n_layers, s);
    default: return launch_wide_hd<0, 256>(p, n_layers, s);
  }
}

int wide_blocks_per_cu(const ShapeDev &sh) {
  if (!wide_available(sh)) return 1;
  if (sh.kv_q8) {
    switch (sh.head_dim) {
      case 64: return wide_occupancy_hd<1, 64>(sh);
      case 128: return wide_occupancy_hd<1, 128>(sh);
      default: return wide_occupancy_hd<1, 256>(sh);
    }
  }
  switch (sh.head_dim) {
    case 64: return wide_occupancy_hd<0, 64>(sh);
    case 128: return wide_occupancy_hd<0, 128>(sh);
    default: return wide_occupancy_hd<0, 256>(sh);
  }
}

}  // namespace g2b
