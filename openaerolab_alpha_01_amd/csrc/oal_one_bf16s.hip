// The one-cell-per-lane step kernel of the bf16s storage form (templates in oal_step_one.h).
#include "oal_step_one.h"

namespace oal {

void launch_one_bf16s(bool wale, const StepArgs& a, hipStream_t stream) { launch_one_sp<StBF16S>(wale, a, stream); }

}  // namespace oal
