// tg_forward_few.hip -- instances of the forward kernels for launches with few workgroups (tg_forward_few.hpp, and those with all of
// a candidate list's places in LDS), without triangles' records.
#include "tg_forward_few.hpp"

namespace tg {

#ifdef TG_DOUBLE_PRECISION
ForwardKernel tile_order_few_kernel() { return nullptr; }
ForwardKernel pixel_order_few_kernel(bool) { return nullptr; }
ForwardKernel pixel_order_helping_kernel(bool) { return nullptr; }
#else
ForwardKernel tile_order_few_kernel() { return forward_tile_order_few_kernel<false>; }
ForwardKernel pixel_order_few_kernel(bool in_turn) {
    return in_turn ? forward_pixel_order_kernel<kSelectBatchShort, uint16_t, true, kLayers, false>
                   : forward_pixel_order_kernel<kSelectBatchShort, uint16_t, false, kLayers, false>;
}
ForwardKernel pixel_order_helping_kernel(bool all_places) {
    return all_places ? forward_pixel_order_helping_kernel<kLayers, false> : forward_pixel_order_helping_kernel<kShortHead, false>;
}
#endif

}  // namespace tg
