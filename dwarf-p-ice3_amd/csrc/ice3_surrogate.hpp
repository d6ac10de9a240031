// ice3_surrogate.hpp -- the surrogate step's network stage (ice3_surrogate.hip).
#pragma once
#include "ice3_stages.hpp"

namespace ice3 {

// Workgroups of the network stage at most, each with a queue segment of its own: a fixed count, so
// that the scratch depends on the problem only.  SG_PARTS wavefronts of the fallback share a segment.
constexpr unsigned int SG_BLOCKS = 256, SG_PARTS = 12;

struct SurrogateArgs {
  MicroArgs m;
  unsigned int npts;                 // nlev * ncol; point q = k * ncol + i
  const ice3_surrogate_norm *norm;
  float budget_tol, neg_tol;
  const void *wpk;                   // packed bf16 weights
  const float *params;               // fp32 parameters (biases)
  unsigned int *queue;               // rejected points' offsets, a segment of seg per workgroup
  unsigned int *qcount;              // their number per workgroup
  unsigned int seg;
  unsigned long long *counters;      // 5 entries, see include/ice3.h
};

__device__ __forceinline__ size_t point_offset(const MicroArgs &m, unsigned int q) {
  return (size_t)(q / m.ncol) * m.ld + q % m.ncol;
}

// Sets a.seg, launches the stage over ncu compute units and returns its number of workgroups (queue
// segments) in nseg.
hipError_t surrogate_network_launch(SurrogateArgs &a, int ncu, unsigned int *nseg, hipStream_t s);

}  // namespace ice3
