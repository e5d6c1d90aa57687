// The one-cell-per-lane FP64 step kernel (templates in oal_step_one.h).
#include "oal_step_one.h"

namespace oal {

void launch_one_f64(bool wale, const TwoRec* rec, uint32_t n, const StepArgs& a, hipStream_t stream) {
    if (!n) return;
    StepArgs r = a;
    r.rec = rec;
    const dim3 g(n * PLANES);
    auto go = [&](auto unit, auto w) {
        constexpr bool U = decltype(unit)::value, W = decltype(w)::value;
        if (a.cp.limiter == 2) hipLaunchKernelGGL((k_step_one<U, W, true>), g, dim3(WG), 0, stream, r);
        else hipLaunchKernelGGL((k_step_one<U, W, false>), g, dim3(WG), 0, stream, r);
    };
    auto rates = [&](auto w) {
        if (a.cp.unit) go(std::true_type{}, w);
        else go(std::false_type{}, w);
    };
    if (wale) rates(std::true_type{});
    else rates(std::false_type{});
}

}  // namespace oal
