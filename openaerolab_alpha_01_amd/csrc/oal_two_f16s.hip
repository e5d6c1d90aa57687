// The two-cells-per-lane step kernel of the f16s storage form (templates in oal_step_two.h).
#include "oal_step_two.h"

namespace oal {

void launch_two_f16s(bool wale, int extra, const StepArgs& a, hipStream_t stream) { launch_two_sp<StF16S>(wale, extra, a, stream); }

}  // namespace oal
