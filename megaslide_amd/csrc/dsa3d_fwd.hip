// Launch of the attention forward for head sizes 32, 64, 96 and 128 (dsa3d_fwd.h).
#include "dsa3d_fwd.h"

namespace msd {

hipError_t launch_dsa3d_fwd_tiled(const msd_dsa3d_desc& d, const void* q, const void* k,
                                  const void* v, const void* off, const void* ek, const void* ev,
                                  void* out, float* lse, hipStream_t s) {
  const Args a = make_tiled_args(d, q, k, v, off, tile_count<1>(d.B, d.T, d.H, d.W), ek, ev);
  if (d.dtype == MSD_BF16) return fwd_typed<bf16, bf16, false>(d, a, out, lse, s);
  return fwd_typed<float, float, false>(d, a, out, lse, s);
}

}  // namespace msd
