// The one-cell-per-lane step kernel of the f32 storage form (templates in oal_step_one.h).
#include "oal_step_one.h"

namespace oal {

void launch_one_f32(bool wale, const StepArgs& a, hipStream_t stream) { launch_one_sp<StF32>(wale, a, stream); }

}  // namespace oal
