// ice3_sedim.hpp -- launch of the statistical sedimentation kernel k_sedim (ice3_sedim.hip).
#pragma once
#include "ice3_stages.hpp"

namespace ice3 {

// Columns per compute unit from which one thread per column, walking it, is the better form:
// of ICE_ADJUST and the sedimentation together (FP64), and of the sedimentation of the mixed
// path.
constexpr int SEDIM_WALK_COLS = 432;

// ICE4_SEDIMENTATION_STAT of the columns of sa with rates in R (double, or float for the mixed
// path) on a device of ncu compute units.  sa.zzz selects the OCND2 model level height and sa.src_rh hail (both FP64).
template <class R> hipError_t sedim_launch(const SedimArgs &sa, int ncu, hipStream_t s);

}  // namespace ice3
