// tg_backward_packed.hip -- the backward kernels' instances that read triangles' records.
#include "tg_backward.hpp"

namespace tg {

#ifdef TG_DOUBLE_PRECISION
BackwardKernel packed_tile_order_backward(GradLayout, bool) { return nullptr; }
BackwardKernel packed_saved_order_backward(GradLayout, bool) { return nullptr; }
#else
BackwardKernel packed_tile_order_backward(GradLayout layout, bool depth) {
    if (layout == kGradBlock8) return depth ? backward_tile_order_kernel<kGradBlock8, true, true> : backward_tile_order_kernel<kGradBlock8, false, true>;
    return depth ? backward_tile_order_kernel<kGradDense, true, true> : backward_tile_order_kernel<kGradDense, false, true>;
}
BackwardKernel packed_saved_order_backward(GradLayout layout, bool depth) {
    if (layout == kGradBlock8) return depth ? backward_saved_order_kernel<kGradBlock8, true, true> : backward_saved_order_kernel<kGradBlock8, false, true>;
    return depth ? backward_saved_order_kernel<kGradDense, true, true> : backward_saved_order_kernel<kGradDense, false, true>;
}
#endif

}  // namespace tg
