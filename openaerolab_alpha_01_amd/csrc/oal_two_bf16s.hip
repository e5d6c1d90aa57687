// The two-cells-per-lane step kernel of the bf16s storage form (templates in oal_step_two.h).
#include "oal_step_two.h"

namespace oal {

void launch_two_bf16s(bool wale, int extra, const StepArgs& a, hipStream_t stream) { launch_two_sp<StBF16S>(wale, extra, a, stream); }

}  // namespace oal
