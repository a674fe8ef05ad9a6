// tg_backward.hip -- launches of the backward kernels (tg_backward.hpp), and their instances without triangles' records.
#include "tg_backward.hpp"

namespace tg {

// The three gradient arrays out of the (V,8) block the per-pixel-order kernels accumulate into:
// one read of the block instead of the three strided ones that three separate copies make.
__global__ __launch_bounds__(256) void split_gradient_block_kernel(const real4 *__restrict__ block, int64_t n_vertices, int copies,
                                                                   real4 *__restrict__ grad_vertices, real *__restrict__ grad_colors,
                                                                   real *__restrict__ grad_opacities) {
    const int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (v >= n_vertices) return;
    real4 position = block[2 * v], rest = block[2 * v + 1];
    for (int k = 1; k < copies; k++) {
        const real4 a = block[2 * (v + k * n_vertices)], b = block[2 * (v + k * n_vertices) + 1];
        position.x += a.x; position.y += a.y; position.w += a.w;
        rest.x += b.x; rest.y += b.y; rest.z += b.z; rest.w += b.w;
    }
    grad_vertices[v] = position;
    grad_colors[3 * v] = rest.x;
    grad_colors[3 * v + 1] = rest.y;
    grad_colors[3 * v + 2] = rest.z;
    grad_opacities[v] = rest.w;
}

size_t backward_pixel_order_lds_bytes(int n_threads) { return pixel_order_lds_bytes(n_threads, kBatch) + (size_t)kAccWindow * kTerms * sizeof(real); }

}  // namespace tg

using namespace tg;

// Waves of a workgroup of the tile-order and the saved-order kernel.  One, but for a frame whose waves all run at once (4096 at most, four
// for each of 1024 SIMDs) and fill a last layer of the SIMDs to more than three quarters: single waves go two to one SIMD and none to the
// next, those of a workgroup of four one to each, which counts where it makes the layers one less.  us, singly and in fours, saved
// order (with a gradient of the depth): 512 x 512 pixels (4096 waves) 248, 231 and 560, 551, 376 x 309 (1920) 230, 217 (251, 234), 256 x 256
// (1024) 430, 421 (484, 462); tile order, 512 x 512 232, 224, 256 x 256 109, 104.  Else: 448 x 448 (3136) 222, 228, 480 x 480 (3600)
// 239, 231 and 576, 596, 362 x 362 (2116) 503, 520 (563, 581), 300 x 300 (1444) 168, 171, 528 x 528 (4356) 259, 262 and 571, 604.
static int workgroup_waves(int width, int height, int tile_w, int tile_h) {
    constexpr int64_t kSimds = 1024;
    const int64_t waves = (int64_t)ceil_div(width, tile_w) * ceil_div(height, tile_h) * ceil_div(tile_w * tile_h, kWave);
    return waves <= 4 * kSimds && (waves - 1) % kSimds >= kSimds / 4 * 3 ? kMaxWaves : 1;
}

int tg::render_backward(const real *grad_image, const real *grad_depthmap, const real *vertices,
                                  const int32_t *indices, const real *colors, const real *opacities,
                                  const int32_t *sorted_ids, const int32_t *offsets, const real *bary, const real *image,
                                  const real *depthmap, const real *final_weights, const int32_t *ends, const int32_t *last,
                                  const real *last_depth, const OrderStore &order, const uint64_t *hit_masks, int width,
                                  int height, int tile_w,
                                  int tile_h, real early_stopping_threshold, int per_pixel_sort, int max_layers, real *grad_vertices,
                                  real *grad_colors, real *grad_opacities, int vertex_stride, int color_stride,
                                  int opacity_stride, int64_t copy_stride, const uint32_t *list_status, int64_t n_keys, const real4 *records, void *stream) {
    if (int e = check_raster_args("tg_render_backward", width, height, tile_w, tile_h, max_layers)) return e;
    if (!grad_image || !vertices || !indices || !colors || !opacities || !offsets || !bary || !image ||
        !depthmap || !final_weights || !ends || !last || !grad_vertices || !grad_colors || !grad_opacities ||
        (per_pixel_sort && !last_depth && !order.low)) {
        set_error("tg_render_backward: null pointer");
        return TG_E_ARG;
    }
    if (vertex_stride < 4 || color_stride < 3 || opacity_stride < 1) {
        set_error("tg_render_backward: gradient strides must be at least 4, 3 and 1");
        return TG_E_ARG;
    }
    if (((uintptr_t)vertices & 15) || ((uintptr_t)image & 15) || ((uintptr_t)grad_image & 15)) {
        set_error("tg_render_backward: vertices, image and grad_image must be 16-byte aligned");
        return TG_E_ARG;
    }
    RasterArgs a{(const real4 *)vertices, indices, colors, opacities, sorted_ids, offsets, bary, nullptr, nullptr,
                 width, height, tile_w, tile_h, early_stopping_threshold, max_layers, kPacks ? records : nullptr};
    const TileLaunch forward = tile_launch(width, height, tile_w, tile_h, kTileThreads);  // whose hit masks are read
    BackwardArgs g{(const real4 *)grad_image, grad_depthmap, (const real4 *)image, depthmap, final_weights, ends, last,
                   last_depth, order, per_pixel_sort ? nullptr : hit_masks, grad_vertices, grad_colors, grad_opacities,
                   vertex_stride, color_stride, opacity_stride, list_status, (int)forward.grid.z, forward.threads, copy_stride,
                   max_layers >= kManyLayers && n_keys / kDeepLists >= (int64_t)ceil_div(width, tile_w) * ceil_div(height, tile_h)};
    hipStream_t s = (hipStream_t)stream;
    const GradLayout layout = (vertex_stride == 4 && color_stride == 3 && opacity_stride == 1)   ? kGradDense
                       : (vertex_stride == 8 && color_stride == 8 && opacity_stride == 8) ? kGradBlock8
                                                                                          : kGradStrided;
#define TG_LAUNCH_BACKWARD(kernel, grid, block, lds_bytes, ...)                                                                              \
    do {                                                                                                                                     \
        if (layout == kGradDense) TG_LAUNCH_AS(#kernel, (kernel<kGradDense __VA_OPT__(,) __VA_ARGS__>), grid, block, lds_bytes, s, a, g);          \
        else if (layout == kGradBlock8) TG_LAUNCH_AS(#kernel, (kernel<kGradBlock8 __VA_OPT__(,) __VA_ARGS__>), grid, block, lds_bytes, s, a, g);   \
        else TG_LAUNCH_AS(#kernel, (kernel<kGradStrided __VA_OPT__(,) __VA_ARGS__>), grid, block, lds_bytes, s, a, g);                             \
    } while (0)
    const TileLaunch waves = tile_launch(width, height, tile_w, tile_h, workgroup_waves(width, height, tile_w, tile_h) * kWave);
    if (!per_pixel_sort) {
        const size_t lds = sizeof(TileWave) * (waves.threads / kWave);
        if (a.records) TG_LAUNCH_AS("backward_tile_order_kernel", packed_tile_order_backward(layout, grad_depthmap != nullptr), waves.grid, dim3(waves.threads), lds, s, a, g);
        else if (grad_depthmap) TG_LAUNCH_BACKWARD(backward_tile_order_kernel, waves.grid, dim3(waves.threads), lds, true, false);
        else TG_LAUNCH_BACKWARD(backward_tile_order_kernel, waves.grid, dim3(waves.threads), lds, false, false);
        return check_launch("backward_tile_order_kernel");
    }
    if (order.low) {
        const size_t lds = sizeof(SavedWave) * (waves.threads / kWave);
        if (a.records) TG_LAUNCH_AS("backward_saved_order_kernel", packed_saved_order_backward(layout, grad_depthmap != nullptr), waves.grid, dim3(waves.threads), lds, s, a, g);
        else if (grad_depthmap) TG_LAUNCH_BACKWARD(backward_saved_order_kernel, waves.grid, dim3(waves.threads), lds, true, false);
        else TG_LAUNCH_BACKWARD(backward_saved_order_kernel, waves.grid, dim3(waves.threads), lds, false, false);
        return check_launch("backward_saved_order_kernel");
    }
    const TileLaunch tl = tile_launch(width, height, tile_w, tile_h, pixel_order_threads(kTileThreads));
    const size_t lds = backward_pixel_order_lds_bytes(tl.threads);
    static size_t lds_reserved[3][kMaxDevices] = {{0}};
    int which = 0;
    for (const void *kernel : {(const void *)backward_pixel_order_kernel<kGradDense>, (const void *)backward_pixel_order_kernel<kGradBlock8>,
                               (const void *)backward_pixel_order_kernel<kGradStrided>})
        if (int e = reserve_lds("tg_render_backward", kernel, lds, lds_reserved[which++])) return e;
    TG_LAUNCH_BACKWARD(backward_pixel_order_kernel, tl.grid, dim3(tl.threads), lds);
    return check_launch("backward_pixel_order_kernel");
#undef TG_LAUNCH_BACKWARD
}

extern "C" int tg_render_backward(const real *grad_image, const real *grad_depthmap, const real *vertices,
                                  const int32_t *indices, const real *colors, const real *opacities,
                                  const int32_t *sorted_ids, const int32_t *offsets, const real *bary, const real *image,
                                  const real *depthmap, const real *final_weights, const int32_t *ends, const int32_t *last,
                                  const real *last_depth, const uint16_t *fragments, const uint64_t *hit_masks, int width,
                                  int height, int tile_w, int tile_h, real early_stopping_threshold, int per_pixel_sort, int max_layers,
                                  real *grad_vertices, real *grad_colors, real *grad_opacities, int vertex_stride, int color_stride,
                                  int opacity_stride, void *stream) {
    if (fragments && per_pixel_sort && max_layers > TG_MAX_SAVED_LAYERS) {
        set_error("tg_render_backward: saved fragments need max_layers <= %d", TG_MAX_SAVED_LAYERS);
        return TG_E_ARG;
    }
    const OrderStore order{const_cast<uint16_t *>(fragments), (int64_t)max_layers * width * height, 0};
    return render_backward(grad_image, grad_depthmap, vertices, indices, colors, opacities, sorted_ids, offsets, bary, image, depthmap,
                           final_weights, ends, last, last_depth, order, hit_masks, width, height, tile_w, tile_h,
                           early_stopping_threshold, per_pixel_sort, max_layers, grad_vertices, grad_colors, grad_opacities,
                           vertex_stride, color_stride, opacity_stride, 0, nullptr, 0, nullptr, stream);
}

extern "C" int tg_render_backward_pooled(const real *grad_image, const real *grad_depthmap, const real *vertices,
                                         const int32_t *indices, int32_t n_triangles, const real *colors, const real *opacities,
                                         const int32_t *sorted_ids, const int32_t *offsets, int64_t n_keys, const real *bary,
                                         const real *image, const real *depthmap, const real *final_weights, const int32_t *ends,
                                         const int32_t *last, const uint16_t *order_pool, int width, int height, int tile_w, int tile_h,
                                         real early_stopping_threshold, int max_layers, real *grad_vertices, real *grad_colors,
                                         real *grad_opacities, int vertex_stride, int color_stride, int opacity_stride, void *stream) {
    if (!order_pool || n_keys < 0 || n_triangles < 0) {
        set_error("tg_render_backward_pooled: null order pool or negative count");
        return TG_E_ARG;
    }
    const int pixels = order_pool_pixels(tile_w, tile_h);
    const OrderStore order{const_cast<uint16_t *>(order_pool), n_triangles > kShortList ? n_keys * pixels : 0, pixels};
    return render_backward(grad_image, grad_depthmap, vertices, indices, colors, opacities, sorted_ids, offsets, bary, image, depthmap,
                           final_weights, ends, last, nullptr, order, nullptr, width, height, tile_w, tile_h, early_stopping_threshold,
                           1, max_layers, grad_vertices, grad_colors, grad_opacities, vertex_stride, color_stride, opacity_stride, 0, nullptr, n_keys, nullptr, stream);
}

extern "C" int tg_split_gradient_block(const real *block, int64_t n_vertices, real *grad_vertices, real *grad_colors,
                                       real *grad_opacities, void *stream) {
    return split_gradient_block(block, n_vertices, 1, grad_vertices, grad_colors, grad_opacities, stream);
}

int tg::split_gradient_block(const real *block, int64_t n_vertices, int copies, real *grad_vertices, real *grad_colors, real *grad_opacities,
                             void *stream) {
    if (n_vertices < 0 || n_vertices > (int64_t)0x7fffffff * 256) {
        set_error("tg_split_gradient_block: n_vertices out of range");
        return TG_E_ARG;
    }
    if (n_vertices == 0) return 0;
    if (!block || !grad_vertices || !grad_colors || !grad_opacities) {
        set_error("tg_split_gradient_block: null pointer");
        return TG_E_ARG;
    }
    if (((uintptr_t)block & 15) || ((uintptr_t)grad_vertices & 15)) {
        set_error("tg_split_gradient_block: block and grad_vertices must be 16-byte aligned");
        return TG_E_ARG;
    }
    TG_LAUNCH(split_gradient_block_kernel, dim3((unsigned)ceil_div64(n_vertices, 256)), dim3(256), 0, (hipStream_t)stream,
              (const real4 *)block, n_vertices, copies, (real4 *)grad_vertices, grad_colors, grad_opacities);
    return check_launch("split_gradient_block_kernel");
}
