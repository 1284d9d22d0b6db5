// G2 constant-work fold on Fm2i: see msm_accum.cuh.
#include "msm_accum.cuh"

namespace g16 {

template <>
void ConstTail<Fm2i>::fold(const ConstJobs& jobs, size_t nseg, int n, hipStream_t s) {
  tail_fold_const<Fm2i>(jobs, nseg, n, s);
}

}  // namespace g16
