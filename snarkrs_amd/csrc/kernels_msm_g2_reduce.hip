// G2 constant-work window reduction on Fm2i: see msm_accum.cuh.
#include "msm_accum.cuh"

namespace g16 {

template <>
void ConstTail<Fm2i>::reduce(const MsmPlan& p, const AccumPtrs& a, uint32_t B, void* window_out,
                             hipStream_t s) {
  tail_reduce_ops<Fm2i, COps<Fm2i>>(p, a, B, window_out, s);
}

}  // namespace g16
