// The two-cells-per-lane step kernel of the f32 storage form (templates in oal_step_two.h).
#include "oal_step_two.h"

namespace oal {

void launch_two_f32(bool wale, int extra, const StepArgs& a, hipStream_t stream) { launch_two_sp<StF32>(wale, extra, a, stream); }

}  // namespace oal
