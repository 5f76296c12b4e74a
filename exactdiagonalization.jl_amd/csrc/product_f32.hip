// The product kernels for one vector type (one translation unit per type: they
// compile side by side).
#include "product.hpp"

namespace edhip {

hipError_t launch_product_f32(const OpDev& op, int transpose, int accumulate, const void* x, void* y, hipStream_t st) {
  return launch_mv_v<float>(op, transpose, accumulate, x, y, st);
}

}  // namespace edhip
