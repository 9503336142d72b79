// Instantiations of the affine prefill kernel for head dim 512 (the f16
// variant decodes the widths that decode_wide_kernel does not take).
#include "prefill_affine.hpp"

namespace tqkv {
namespace prefill {
KernelFn pick_d512(int bk, int bv, bool h16) {
  return h16 ? pick_for<512, true>(bk, bv) : pick_for<512, false>(bk, bv);
}
}  // namespace prefill
}  // namespace tqkv
