// The one-cell-per-lane step kernel of the f64 storage form (templates in oal_step_one.h).
#include "oal_step_one.h"

namespace oal {

void launch_one_f64(bool wale, bool wide, const StepArgs& a, hipStream_t stream) { launch_one_sp<StF64>(wale, a, stream, wide); }

}  // namespace oal
