// bf16 instantiation of the fused MLP kernels (templates in mlp16.h).
#include "mlp16.h"

namespace srf {
namespace mlp {

int fwd_bf16(const FwdArgs& a, bool vd, bool tr, hipStream_t s) {
  if (tr) return vd ? launch_fwd16<kBF16, true, true, 2>(a, s) : launch_fwd16<kBF16, false, true, 2>(a, s);
  return vd ? launch_infer16<kBF16, true>(a, s) : launch_infer16<kBF16, false>(a, s);
}

int bwd_bf16(const BwdArgs& a, bool vd, hipStream_t s) {
  return vd ? launch_bwd16<kBF16, true>(a, s) : launch_bwd16<kBF16, false>(a, s);
}

}  // namespace mlp
}  // namespace srf
