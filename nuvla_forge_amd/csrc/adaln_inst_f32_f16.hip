// adaLN row kernels instantiated for x = float, y = f16.
#include "adaln_impl.h"

namespace nf {
namespace adaln {
template int fwd_v<float, f16>(const FwdArgs &, const Plan &, bool, hipStream_t);
template int bwd_v<float, f16>(const BwdArgs &, const Plan &, bool, hipStream_t);
template int bwd_walk<float, f16>(const BwdArgs &, const WalkOut &, const Plan &,
                                 const WalkPlan &, hipStream_t);
}  // namespace adaln
}  // namespace nf
