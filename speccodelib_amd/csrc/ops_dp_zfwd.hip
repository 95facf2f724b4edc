// FP64 instances of the fused z-forward.
#define SCL_OPS_ZFWD
#include "ops_impl.hpp"
namespace scl {
template int32_t Ops<double>::zfwd_rhs(const scl_plan3d&, int, cpx<double>*, int64_t, cpx<double>*, cpx<double>*, cpx<double>*,
                                        const cpx<double>*, const double*, const RhsParams<double>&, bool);
}  // namespace scl
