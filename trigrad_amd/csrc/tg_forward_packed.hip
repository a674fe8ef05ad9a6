// tg_forward_packed.hip -- the forward kernels' instances that read triangles' records.
#include "tg_forward_few.hpp"

namespace tg {

#ifdef TG_DOUBLE_PRECISION
ForwardKernel packed_tile_order_kernel() { return nullptr; }
ForwardKernel packed_tile_order_few_kernel() { return nullptr; }
ForwardKernel packed_pixel_order_kernel(bool, bool, bool) { return nullptr; }
ForwardKernel packed_pixel_order_bounds_kernel(bool) { return nullptr; }
LongListsKernel packed_pixel_order_long_lists_kernel() { return nullptr; }
#else
ForwardKernel packed_tile_order_kernel() { return forward_tile_order_kernel<true>; }
ForwardKernel packed_tile_order_few_kernel() { return forward_tile_order_few_kernel<true>; }
ForwardKernel packed_pixel_order_kernel(bool tiles_help, bool all_places, bool in_turn) {
    if (tiles_help) return all_places ? forward_pixel_order_helping_kernel<kLayers, true> : forward_pixel_order_helping_kernel<kShortHead, true>;
    if (all_places)
        return in_turn ? forward_pixel_order_kernel<kSelectBatchShort, uint16_t, true, kLayers, true>
                       : forward_pixel_order_kernel<kSelectBatchShort, uint16_t, false, kLayers, true>;
    return in_turn ? forward_pixel_order_kernel<kSelectBatchShort, uint16_t, true, kShortHead, true>
                   : forward_pixel_order_kernel<kSelectBatchShort, uint16_t, false, kShortHead, true>;
}
ForwardKernel packed_pixel_order_bounds_kernel(bool in_turn) {
    return in_turn ? forward_pixel_order_kernel<kSelectBatch, int, true, kLayers, true> : forward_pixel_order_kernel<kSelectBatch, int, false, kLayers, true>;
}
LongListsKernel packed_pixel_order_long_lists_kernel() { return forward_pixel_order_long_lists_kernel<true>; }
#endif

}  // namespace tg
