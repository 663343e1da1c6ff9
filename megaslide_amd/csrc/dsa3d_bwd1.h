// Launch of the first backward kernel (dsa3d_bwd1.hip; instantiated there).
#pragma once

#include "dsa3d_tiled_common.h"

namespace msd {

template <int HD, typename E, int AE, bool REC, bool SPLIT = false>
void launch_bwd_p1(const tiled::Args& a, const E* dout, const float* lse, const float* dlse, E* doff,
                   float* p_ws, float* b_ws, void* dk_acc, void* dv_acc, int64_t acc_ks,
                   int64_t acc_vs, const tiled::RecArgs& rc, hipStream_t s);

}  // namespace msd
