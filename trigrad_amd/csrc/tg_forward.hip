// tg_forward.hip -- forward rasterize-and-blend, one workgroup per tile.
//
// per_pixel_sort = 0 (tile order): the sorted tile list is staged into LDS in
//   batches of 128 records; each pixel composites front to back and stops as
//   soon as its transmittance falls to the threshold or max_layers fragments
//   are blended; the workgroup leaves the list when every pixel has stopped.
// per_pixel_sort = 1: each pixel repeatedly selects its next (up to 32) nearest
//   fragments in (pixel depth, list position) order by scanning the whole list
//   (records staged through LDS as above, candidate lists in LDS, slot-major),
//   then blends them; threshold and max_layers are tested between selections
//   only, as in the reference (render.cu:588).
//
// Not HBM-bound: per (pixel, entry) pair ~12 VALU operations and three
// broadcast LDS reads against 148 B of gathered data per ENTRY.
#include <algorithm>

#include "tg_forward_pixel.hpp"

namespace tg {

// Workgroups for the long tiles where they are shared out, at most: as many as run at once, four a CU; fewer may find too much
// (1920 x 1080, 200 tiles of 1100 large faint triangles among 60 000 small ones, forward, us: 128 workgroups 630, 512 396, 1024
// 339, one for each tile 478; without a limit on the layers 1597, 890, 637, 1048; 54 tiles of 32 x 32 in tile order, 256 210, 512
// 158, 1024 110).  Those that find nothing cost nothing that shows: 10^6 triangles 671 with 128 and 670 with 1024, 10^5 253 and
// 254, a mesh of 1.3 million 716 and 718.  They do where there is one generation of workgroups, which in per-pixel order therefore
// has the places that are left and at least 128 of them, and help from the tiles' own (forward_pixel_order_helping_kernel; depth
// bounds, where two workgroups run on a CU, keep to the many in front: 200 000 faint triangles 845 us, with help 850), and in tile
// order, from 257 workgroups on, half as many (400 tiles with lists of 1000 large faint triangles, frames, us: 246, with 1024 275; 576
// with 350, 184 and 196; 1024 tiles, 100 of them with 3000, 497 and 496).
constexpr int kLongGroups = 1024, kLongGroupsTileOrder = 512;
TileLaunch tile_launch(int width, int height, int tile_w, int tile_h, int max_threads) {
    TileLaunch t;
    const int pixels = tile_w * tile_h;
    t.threads = min(ceil_div(pixels, kWave) * kWave, max_threads);
    t.grid = dim3(ceil_div(width, tile_w), ceil_div(height, tile_h), ceil_div(pixels, t.threads));
    return t;
}

// Workgroup size of the per-pixel-sort kernels: the 256 threads of a 16x16 tile.  They are bound by latency, so what counts is
// how many waves a CU holds, and that is set by the candidate lists in LDS.  With int positions (depth bounds, longest lists,
// and the re-selecting backward kernel, which also keeps 43 KB of gradient sums) those take 32 * (scalar + int) bytes a thread,
// 64 KB a workgroup, two a CU next to 128 staged entries (8 KB); with 16-bit positions 48 KB, three, or 34.5 KB with 23
// places, four (candidate_places).  Measured with int positions on frames of all sizes against 64, 192 and 256 staged entries
// and against tiles split over two workgroups of 128 threads or four of 64 (which stage every entry two or four times): 15 to
// 35 % faster than 256 entries and 128 threads.
// TRIGRAD_PIXEL_ORDER_THREADS (64, 128 or 256) overrides the workgroup size.
int pixel_order_threads(int preferred) {
    static int override = -1;
    if (override < 0) {
        override = 0;
        if (const char *e = getenv("TRIGRAD_PIXEL_ORDER_THREADS")) {
            const int x = atoi(e);
            if (x == 64 || x == 128 || x == 256) override = x;
        }
    }
    return override ? override : preferred;
}

size_t pixel_order_lds_bytes(int n_threads, int staged_entries, size_t position_bytes, int places) {
    return sizeof(DepthRecord) * staged_entries + (size_t)places * n_threads * (sizeof(real) + position_bytes);
}

// Places of a pixel's candidate list that a launch with 16-bit positions keeps in LDS: kShortHead or all.
// Short heads are worth it where they save a generation of workgroups (four a CU in the place of three, or eleven of a wave in
// the place of nine).  Where they do not, the kernel is the same number of latency chains after one another, which the tail
// and its single records lengthen.  Per-pixel order, frames in us with all places and with short heads: 323 tiles of 8 x 8
// with 240 small faint triangles each, one generation of either, kernel 47 and 51; 1224 tiles of 16 x 16, two of either, 213 and
// 230; 2074, three of either, 347 and 385; 3480 of 8 x 8, two of either, 250 and 275.  1000 tiles, two and one, 154 and 139;
// 3773, five and four, 302 and 281; 2646 of 8 x 8, two and one, 148 and 133.
static int candidate_places(int64_t groups, int n_threads) {
    const auto generations = [&](int places) {  // LDS comes in pieces of 1280 bytes
        const int64_t pieces = ceil_div64((int64_t)pixel_order_lds_bytes(n_threads, kSelectBatchShort, sizeof(uint16_t), places) + 512, 1280);
        return ceil_div64(groups, 256 * std::min<int64_t>(short_list_waves(places) * kTileThreads / n_threads, 128 / pieces));
    };
    return generations(kLayers) <= generations(kShortHead) ? kLayers : kShortHead;
}

int check_raster_args(const char *fn, int width, int height, int tile_w, int tile_h, int max_layers) {
    if (width <= 0 || height <= 0 || tile_w <= 0 || tile_h <= 0 || tile_w * tile_h > kMaxTilePixels) {
        set_error("%s: image size must be positive and tile_w*tile_h in [1, %d]", fn, kMaxTilePixels);
        return TG_E_ARG;
    }
    if ((int64_t)width * height > 0x7fffffffll) {
        set_error("%s: image too large", fn);
        return TG_E_ARG;
    }
    if (max_layers <= 0) {
        set_error("%s: max_layers must be positive", fn);
        return TG_E_ARG;
    }
    return 0;
}

}  // namespace tg

using namespace tg;

extern "C" int tg_candidate_places(int width, int height, int tile_w, int tile_h) {
    if (width <= 0 || height <= 0 || tile_w <= 0 || tile_h <= 0 || tile_w * tile_h > kMaxTilePixels) return 0;
    const TileLaunch tl = tile_launch(width, height, tile_w, tile_h, pixel_order_threads(kTileThreads));
    return candidate_places((int64_t)tl.grid.x * tl.grid.y * tl.grid.z, tl.threads);
}

extern "C" size_t tg_hit_mask_words(int64_t n_keys, int width, int height, int tile_w, int tile_h) {
    if (n_keys < 0 || width <= 0 || height <= 0 || tile_w <= 0 || tile_h <= 0 || tile_w * tile_h > kMaxTilePixels) return 0;
    const TileLaunch tl = tile_launch(width, height, tile_w, tile_h, kTileThreads);
    const int64_t tiles = (int64_t)tl.grid.x * tl.grid.y;
    return (size_t)(tiles * tl.grid.z + (n_keys / kWave + tiles + 1) * (int64_t)tl.grid.z * tl.threads);
}

int tg::render_forward(const real *vertices, const int32_t *indices, const real *colors, const real *opacities,
                                 const int32_t *sorted_ids, const int32_t *offsets, const real *bary, int width, int height,
                                 int tile_w, int tile_h, real early_stopping_threshold, int per_pixel_sort, int max_layers,
                                 real *image, real *depthmap, real *final_weights, int32_t *ends, int32_t *last,
                                 real *last_depth, const OrderStore &order, uint64_t *hit_masks, const real *batch_bounds,
                                 const int32_t *far_start, const uint32_t *list_status, uint32_t *host_status, int64_t longest,
                                 const LongTiles &long_tiles, const real4 *records, void *stream) {
    if (int e = check_raster_args("tg_render_forward", width, height, tile_w, tile_h, max_layers)) return e;
    if (!vertices || !indices || !colors || !opacities || !offsets || !bary || !image || !depthmap || !final_weights || !ends) {
        set_error("tg_render_forward: null pointer");
        return TG_E_ARG;
    }
    if (((uintptr_t)vertices & 15) || ((uintptr_t)image & 15)) {
        set_error("tg_render_forward: vertices and image must be 16-byte aligned");
        return TG_E_ARG;
    }
    RasterArgs a{(const real4 *)vertices, indices, colors, opacities, sorted_ids, offsets, bary,
                 per_pixel_sort ? batch_bounds : nullptr, (per_pixel_sort && batch_bounds) ? far_start : nullptr,
                 width, height, tile_w, tile_h, early_stopping_threshold, max_layers, kPacks ? records : nullptr};
    const bool packed = a.records != nullptr;
    if (batch_bounds && !far_start) {
        set_error("tg_render_forward: batch_bounds come with far_start");
        return TG_E_ARG;
    }
    ForwardOut o{(real4 *)image, depthmap, final_weights, ends, last, last_depth, order, per_pixel_sort ? nullptr : hit_masks,
                 list_status, host_status, long_tiles, 0};
    const TileLaunch tl = tile_launch(width, height, tile_w, tile_h, per_pixel_sort ? pixel_order_threads(kTileThreads) : kTileThreads);
    const int64_t groups = (int64_t)tl.grid.x * tl.grid.y * tl.grid.z;
    const bool split_tiles = kSharesLongTiles && !per_pixel_sort && tl.threads == kTileThreads && groups <= kFewTileGroups;
    bool tiles_help = false;
    if (long_tiles.words && (per_pixel_sort || split_tiles || groups > 256 * 8)) {  // eight in tile order run on a CU at once: then none is first
        const bool shared_out = per_pixel_sort ? tl.threads == kTileThreads : split_tiles;
        tiles_help = kSharesLongTiles && shared_out && per_pixel_sort && !a.batch_bounds && groups <= kLongGroups;
        int most = kLongGroups;
        if (tiles_help) most = std::max(kLongGroups - (int)groups, kLongTileSlots);
        else if (!shared_out) most = kLongTileSlots;
        else if (!per_pixel_sort && groups > 256) most = kLongGroupsTileOrder;
        o.long_rows = ceil_div((int)std::min<int64_t>(ceil_div(most, (int)tl.grid.z), kMaxTileWaves * long_tiles.most), (int)tl.grid.x);
    }
    const dim3 grid(tl.grid.x, tl.grid.y + o.long_rows, tl.grid.z);
    const int n_threads = tl.threads;
    hipStream_t s = (hipStream_t)stream;
    if (!per_pixel_sort) {
        if (split_tiles)
            TG_LAUNCH_AS("forward_tile_order_few_kernel", packed ? packed_tile_order_few_kernel() : tile_order_few_kernel(), grid, dim3(n_threads), 0, s, a, o);
        else
            TG_LAUNCH_AS("forward_tile_order_kernel", packed ? packed_tile_order_kernel() : forward_tile_order_kernel<false>, grid,
                         dim3(n_threads), 0, s, a, o);
        return check_launch("forward_tile_order_kernel");
    }
    const size_t lds = pixel_order_lds_bytes(n_threads, kSelectBatch);
    static size_t lds_reserved[2][8][kMaxDevices] = {{{0}}}, lds_reserved_long[2][kMaxDevices] = {{0}};
    const bool in_turn = n_threads == kTileThreads;
    const auto launch = [&](void (*kernel)(RasterArgs, ForwardOut), size_t lds_bytes, size_t *reserved) -> int {
        if (int e = reserve_lds("tg_render_forward", (const void *)kernel, lds_bytes, reserved)) return e;
        TG_LAUNCH_AS("forward_pixel_order_kernel", kernel, grid, dim3(n_threads), lds_bytes, s, a, o);
        return check_launch("forward_pixel_order_kernel");
    };
    if (a.batch_bounds)  // they make the batches jump in steps of kSelectBatch
        return launch(packed    ? packed_pixel_order_bounds_kernel(in_turn)
                      : in_turn ? forward_pixel_order_kernel<kSelectBatch, int, true, kLayers, false>
                                : forward_pixel_order_kernel<kSelectBatch, int, false, kLayers, false>, lds, lds_reserved[packed][in_turn]);
    const int places = candidate_places(groups, n_threads);
    const bool all_places = kShortHead < kLayers && places == kLayers;
    const size_t lds_short = pixel_order_lds_bytes(n_threads, kSelectBatchShort, sizeof(uint16_t), places);
    const auto short_kernel = packed       ? packed_pixel_order_kernel(tiles_help, all_places, in_turn)
                              : tiles_help ? pixel_order_helping_kernel(all_places)
                              : all_places ? pixel_order_few_kernel(in_turn)
                              : in_turn    ? forward_pixel_order_kernel<kSelectBatchShort, uint16_t, true, kShortHead, false>
                                           : forward_pixel_order_kernel<kSelectBatchShort, uint16_t, false, kShortHead, false>;
    if (int e = launch(short_kernel, lds_short, lds_reserved[packed][tiles_help ? 6 + all_places : 2 + 2 * all_places + in_turn])) return e;
    // no list is too long for 16-bit positions, or those that are are long tiles, which the kernel above has shared out
    if (longest <= kShortList || (in_turn && o.long_rows && long_tiles.limit <= kShortList)) return 0;
    const auto long_kernel = packed ? packed_pixel_order_long_lists_kernel() : forward_pixel_order_long_lists_kernel<false>;
    if (int e = reserve_lds("tg_render_forward", (const void *)long_kernel, lds, lds_reserved_long[packed])) return e;
    const int tiles = (int)(tl.grid.x * tl.grid.y);
    TG_LAUNCH_AS("forward_pixel_order_long_lists_kernel", long_kernel, dim3(min(tiles, kLongListGroups), 1, grid.z), dim3(n_threads), lds, s, a, o,
                 (int)tl.grid.x, (int)tl.grid.y);
    return check_launch("forward_pixel_order_long_lists_kernel");
}

extern "C" int tg_render_forward(const real *vertices, const int32_t *indices, const real *colors, const real *opacities,
                                 const int32_t *sorted_ids, const int32_t *offsets, const real *bary, int width, int height,
                                 int tile_w, int tile_h, real early_stopping_threshold, int per_pixel_sort, int max_layers,
                                 real *image, real *depthmap, real *final_weights, int32_t *ends, int32_t *last,
                                 real *last_depth, uint16_t *fragments, uint64_t *hit_masks, const real *batch_bounds,
                                 const int32_t *far_start, const uint32_t *list_status, void *stream) {
    if (fragments && (!per_pixel_sort || max_layers > TG_MAX_SAVED_LAYERS)) {
        set_error("tg_render_forward: fragments are saved only with per_pixel_sort and max_layers <= %d", TG_MAX_SAVED_LAYERS);
        return TG_E_ARG;
    }
    const OrderStore order{fragments, (int64_t)max_layers * width * height, 0};
    return render_forward(vertices, indices, colors, opacities, sorted_ids, offsets, bary, width, height, tile_w, tile_h,
                          early_stopping_threshold, per_pixel_sort, max_layers, image, depthmap, final_weights, ends, last, last_depth,
                          order, hit_masks, batch_bounds, far_start, list_status, nullptr, std::numeric_limits<int64_t>::max(), LongTiles(), nullptr, stream);
}

extern "C" int64_t tg_order_pool_words(int64_t n_keys, int64_t n_triangles, int tile_w, int tile_h) {
    if (n_keys < 0 || n_triangles < 0 || tile_w <= 0 || tile_h <= 0 || tile_w * tile_h > kMaxTilePixels) return 0;
    // a triangle is in a tile's list once, so no list is longer than the number of triangles
    return n_keys * order_pool_pixels(tile_w, tile_h) * (n_triangles > kShortList ? 2 : 1);
}

extern "C" int tg_render_forward_pooled(const real *vertices, const int32_t *indices, int32_t n_triangles, const real *colors,
                                        const real *opacities, const int32_t *sorted_ids, const int32_t *offsets, int64_t n_keys,
                                        const real *bary, int width, int height, int tile_w, int tile_h, real early_stopping_threshold,
                                        int max_layers, real *image, real *depthmap, real *final_weights, int32_t *ends, int32_t *last,
                                        real *last_depth, uint16_t *order_pool, const real *batch_bounds, const int32_t *far_start,
                                        const uint32_t *list_status, void *stream) {
    if (!order_pool || n_keys < 0 || n_triangles < 0) {
        set_error("tg_render_forward_pooled: null order pool or negative count");
        return TG_E_ARG;
    }
    const int pixels = order_pool_pixels(tile_w, tile_h);
    const OrderStore order{order_pool, n_triangles > kShortList ? n_keys * pixels : 0, pixels};
    return render_forward(vertices, indices, colors, opacities, sorted_ids, offsets, bary, width, height, tile_w, tile_h,
                          early_stopping_threshold, 1, max_layers, image, depthmap, final_weights, ends, last, last_depth, order, nullptr,
                          batch_bounds, far_start, list_status, nullptr, n_keys, LongTiles(), nullptr, stream);
}
