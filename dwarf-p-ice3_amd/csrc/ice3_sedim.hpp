// ice3_sedim.hpp -- launch of the statistical sedimentation (ice3_sedim.hip).
#pragma once
#include "ice3_stages.hpp"

namespace ice3 {

// ICE4_SEDIMENTATION_STAT of the columns of sa with rates in R (double, or float for the mixed
// path) on a device of ncu compute units.  sa.zzz selects the OCND2 model level height and sa.src_rh hail (both FP64).
template <class R> hipError_t sedim_launch(const SedimArgs &sa, int ncu, hipStream_t s);
template <> hipError_t sedim_launch<double>(const SedimArgs &sa, int ncu, hipStream_t s);
template <> hipError_t sedim_launch<float>(const SedimArgs &sa, int ncu, hipStream_t s);

}  // namespace ice3
