// The product kernels for one vector type (one translation unit per type: they
// compile side by side).
#include "product.hpp"

namespace edhip {

hipError_t launch_product_f64(const OpDev& op, int transpose, int accumulate, const void* x, void* y, hipStream_t st) {
  return launch_mv_v<double>(op, transpose, accumulate, x, y, st);
}

hipError_t launch_window_product_f64(const WinOp& P, int Lx, int Ly, int unit, int transpose, const void* x, void* y,
                                    hipStream_t st) {
  return launch_win_other<double>(P, Lx, Ly, unit, transpose, x, y, st);
}

}  // namespace edhip
