// FP32 instances of the fused z-forward.
#define SCL_OPS_ZFWD
#include "ops_impl.hpp"
namespace scl {
template int32_t Ops<float>::zfwd_rhs(const scl_plan3d&, int, cpx<float>*, int64_t, cpx<float>*, cpx<float>*, cpx<float>*,
                                        const cpx<float>*, const double*, const RhsParams<float>&, bool);
}  // namespace scl
