// qmv_batch_kernel (vpq_qmv_batch.h) for the format twins: 8-bit codes, groups of 32, binary16 elements.
#include "vpq_qmv_batch.h"

namespace vpq {

hipError_t launch_qmv_batch_twin(hipStream_t st, const BatchParams& p, const BatchPlan& plan, size_t lds_bytes, int grid,
                                 const BatchFormat& f)
{
  if (f.bits == 4 && f.group == 64 && f.f16) { return batch_launch<4, 64, true>(st, p, plan, lds_bytes, grid); }
  if (f.bits == 4 && f.group == 32 && !f.f16) {
    return f.scale_only ? batch_launch<4, 32, false, true>(st, p, plan, lds_bytes, grid)
                        : batch_launch<4, 32, false, false>(st, p, plan, lds_bytes, grid);
  }
  if (f.bits == 8 && f.group == 64 && !f.f16) { return batch_launch<8, 64, false>(st, p, plan, lds_bytes, grid); }
  if (f.bits == 8 && f.group == 32 && !f.f16) { return batch_launch<8, 32, false>(st, p, plan, lds_bytes, grid); }
  return hipErrorInvalidValue;
}

}  // namespace vpq
