// tg_frame.hip -- a frame's forward pass, and its backward pass, in one call each.
//
// Small frames are bound by the host: a frame of 20 triangles keeps the GPU busy for 70 us and took 310 us when every stage
// was a call of its own with its own buffers and the host waited for K (the number of keys) half way, to size the rest.
// Here the host launches the whole chain for the capacity of the key buffers, the kernels read K on the device, and the
// host waits for K only when everything is under way: it then knows whether the buffers were large enough (if not, the
// kernels have made empty lists and the caller comes again with larger ones).  K and the list kernels' status word are
// written by the kernels into pinned host memory and found there by looking, so a frame has no copies and no events.
#include <hip/hip_runtime.h>
#include <immintrin.h>

#include <algorithm>
#include <atomic>
#include <chrono>

#include "tg_frame.hpp"
#include "tg_gradient_copies.hpp"

namespace tg {

#ifndef TG_DOUBLE_PRECISION
struct FrameLayout {
    // kept: what the backward pass and the caller look at later
    size_t status, ids, offsets, bary, weights, ends, last, last_depth, order, masks, kept_bytes;
    // scratch: dead when the forward pass is done
    size_t keys, keys_alt, values_alt, sort, long_tiles, all_long_tiles, bounds, far_start, low, scratch_bytes;
    size_t sort_bytes, zero_bytes;  // of the sort's workspace, and what of it (and of the long tiles' count) starts at zero
    int long_limit;                 // list entries that make a tile a long one; 0: the frame has no use for them
};

// Which frames make triangles' records (TriangleRecord).  They cost the scan 20 us for 10^6 triangles, and the passes gain by every list
// entry they read: little where neighbouring triangles share vertices, whose lines they share as well (a mesh of 1.3 million, forward, us, 260
// and 264), where what is read of all triangles is in the L2s anyway, and in tile order, which leaves long lists early.  Soups,
// frames in us, without and with: per-pixel order, train, 50 000 small triangles on 1024 x 1024 135, 135, 10^5 152, 154, 150 000
// 173, 172, 200 000 197, 192, 500 000 347, 329, 10^6 670, 586; shown, 10^5 144, 146, 150 000 168, 168, 300 000 245, 237, 10^6
// 997, 907 (lists of 700).  Tile order, train, 300 000 on 1920 x 1080 247, 251, 500 000 348, 343, 10^6 588, 565 (lists of 270), on 1024 x 1024
// with lists of 400 573, 542, of 700 611, 609, on 512 x 512 with lists of 2000 549, 551, of 2800 393, 419; with a heavy tail of large
// triangles it is about the same, 800 000 on 1920 x 1080 707, 706, 1.2 million 818, 829, 2 million 1030, 1030.
// Tile order, shown: the forward pass alone is to gain what the scan loses.  It does while the scan's workgroups with records are no more
// than the CUs (524 288 triangles), where triangles are so small that lists are walked to their ends (mean edges of 1.5 pixels, 1.19 keys
// a triangle), and from where the arrays are more than the memory-side cache holds, unless large triangles end the walks (2.19 keys).
// 1920 x 1080, mean edges of 1.5, 4, 8 pixels, and of 4 with a heavy tail: 523 000 173, 162 and 193, 190 and 247, 250 and 251, 252; 530 000 179, 176
// and 202, 208 and 255, 264 and 257, 271; 1.2 million 319, 316 and 357, 376 and 432, 470 and 399, 437; 1.6 million 406, 384 and 467, 463 and 583, 585 and
// 494, 518; 1.76 million 454, 415 and 501, 495 and 643, 635 and 534, 552; 2.5 million 647, 560 and 754, 693 and 836, 788 and 662, 683.  (A
// key buffer has room for an eighth and up to a sixteenth more than a frame's keys.)
constexpr int64_t kRecordsTriangles = 150000, kRecordsTrianglesTileOrder = 500000, kRecordsListTileOrder = 800;
constexpr int64_t kShownScanAtOnce = 256 * 2048, kShownBeyondCache = 1700000;
static bool may_have_records(const tg_frame &f) {
    const bool backward_reads_matrices = (f.flags & TG_FRAME_BACKWARD) && f.per_pixel_sort && !(f.flags & (TG_FRAME_ORDER_PLANES | TG_FRAME_ORDER_POOL));
    return (f.flags & TG_FRAME_RECORDS) && f.n_triangles >= (f.per_pixel_sort ? kRecordsTriangles : kRecordsTrianglesTileOrder) && !backward_reads_matrices;
}
// Where a frame's buffers have room for records: wherever it or one of fewer triangles has them.  A mesh, which has none, keeps 36 bytes a
// triangle until its backward pass, and not 128.
static bool has_room_for_records(const tg_frame &f) {
    const int64_t tiles = ceil_div64(f.width, f.tile_w) * ceil_div64(f.height, f.tile_h);
    return may_have_records(f) && f.n_vertices >= 2 * f.n_triangles && (f.per_pixel_sort || f.key_capacity <= kRecordsListTileOrder * tiles);
}
static bool has_records(const tg_frame &f) {
    if (!has_room_for_records(f)) return false;
    const int64_t M = f.n_triangles;
    if (f.per_pixel_sort || (f.flags & TG_FRAME_BACKWARD) || M <= kShownScanAtOnce) return true;
    return 2 * f.key_capacity <= (M < kShownBeyondCache ? 3 * M : 4 * M);
}

// No size is larger for a smaller number of triangles, all else equal: callers size buffers for a rounded one.  (For records that is so
// among numbers of triangles with two vertices or more each, and among those with fewer: a plan is for the one or the other.)
static FrameLayout frame_layout(const tg_frame &f) {
    FrameLayout L = {};
    const int tiles_x = (int)ceil_div64(f.width, f.tile_w), tiles_y = (int)ceil_div64(f.height, f.tile_h), tiles = tiles_x * tiles_y;
    const int64_t pixels = f.width * f.height;
    size_t o = 0;
    const auto take = [&](size_t bytes) { const size_t at = o; o = (o + bytes + 255) & ~(size_t)255; return at; };
    const bool backward = f.flags & TG_FRAME_BACKWARD;
    L.status = take(4);  // of the sort
    L.ids = take((size_t)f.key_capacity * 4);
    L.offsets = take((size_t)(tiles + 1) * 4);
    L.bary = take((size_t)f.n_triangles * (has_room_for_records(f) ? sizeof(TriangleRecord) : 9 * sizeof(real)));  // the records' place is that of the matrices
    L.weights = take((size_t)pixels * sizeof(real));
    L.ends = take((size_t)pixels * 4);
    if (backward) {
        L.last = take((size_t)pixels * 4);
        if (f.per_pixel_sort) L.last_depth = take((size_t)pixels * sizeof(real));
        if (f.flags & TG_FRAME_ORDER_PLANES) L.order = take((size_t)(2 * f.max_layers * pixels) * 2);
        if (f.flags & TG_FRAME_ORDER_POOL)
            L.order = take((size_t)tg_order_pool_words(f.key_capacity, f.n_triangles, (int)f.tile_w, (int)f.tile_h) * 2);
        if (f.flags & TG_FRAME_HIT_MASKS)
            L.masks = take(tg_hit_mask_words(f.key_capacity, (int)f.width, (int)f.height, (int)f.tile_w, (int)f.tile_h) * 8);
    }
    L.kept_bytes = o;
    o = 0;
    L.keys = take((size_t)f.key_capacity * 8);
    L.keys_alt = take((size_t)f.key_capacity * 8);
    L.values_alt = take((size_t)f.key_capacity * 4);
    L.sort_bytes = tg_build_frame_lists_workspace_bytes(f.key_capacity, tiles_x, tiles_y);
    L.sort = take(L.sort_bytes);
    L.zero_bytes = L.sort_bytes;
    // Long: 1024 entries, and twice the mean.  In frames with a workgroup (256 pixels) for half of the CUs at most in per-pixel
    // order, for each CU in tile order, 1024 entries are enough, because much of the chip has nothing else to do -- unless a
    // triangle is in more than four tiles on average: such triangles fill a pixel's layers, and depth bounds end the looking,
    // long before the list does.  Shorter lists are served as well by the others' way.  Forward
    // kernel, us: mesh of 1.3 million triangles, per-pixel order, 1024 entries 333, 768 336, 1400 350; mesh of 800 000 on 42 tiles
    // 4640, with those of twice the mean shared out 2153, with all 1118; 42 tiles with 3200 large triangles each 87, shared out 101.
    // Frames, us, all lists alike, by one workgroup each and shared out, per-pixel order: 96 workgroups with lists of 3500
    // 492, 322; 126 with 6200 727, 406; 132 with 1700 298, 328; 182 with 1400 312, 377; 432 (tiles of 32 x 32) with 2900 314, 790.
    // Tile order: 209 with 3500 189, 167; 238 with 1700 270, 227; 320 (32 x 32) with 3000 129, 149.
    const int64_t longest = f.key_capacity < f.n_triangles ? f.key_capacity : f.n_triangles;
    const int64_t at_once = 256 * (f.per_pixel_sort ? 3 : 8);
    const int64_t groups = (int64_t)tiles * ceil_div64(f.tile_w * f.tile_h, kTileThreads);
    const bool few = groups <= (f.per_pixel_sort ? 128 : 256) && f.key_capacity <= 4 * f.n_triangles;
    const int64_t limit = std::max<int64_t>(1024, few ? 0 : ceil_div64(2 * f.key_capacity, tiles));
    if (longest >= limit) L.long_limit = (int)limit;
    if (L.long_limit || tiles <= at_once) {  // where the place is small, it is there whatever the number of triangles
        L.long_tiles = take((kLongTileCounters + 1 + kLongTileSlots) * 4);
        L.all_long_tiles = take((size_t)tiles * 4);
        L.zero_bytes = L.long_tiles + (kLongTileCounters + 1) * 4 - L.sort;
    }
    if (f.flags & TG_FRAME_LIST_BOUNDS) {
        L.bounds = take(tg_list_bound_words(f.key_capacity, tiles) * sizeof(real));
        L.far_start = take((size_t)tiles * 4);
        L.low = take((size_t)f.n_triangles * sizeof(real));
    }
    L.scratch_bytes = o;
    return L;
}

static int check_frame(const char *fn, const tg_frame *f) {
    if (!f || f->n_vertices < 0 || f->n_vertices > 0x7fffffff || f->n_triangles <= 0 || f->n_triangles > 0x7fffffff || f->width <= 0 ||
        f->height <= 0 || f->width > 0x7fffffff || f->height > 0x7fffffff || f->tile_w <= 0 || f->tile_h <= 0 ||
        f->tile_w > kMaxTilePixels || f->tile_h > kMaxTilePixels || f->key_capacity <= 0 || f->key_capacity >= (1ll << 30)) {
        set_error("%s: null frame, or a size out of range", fn);
        return TG_E_ARG;
    }
    if (int e = check_raster_args(fn, (int)f->width, (int)f->height, (int)f->tile_w, (int)f->tile_h, (int)f->max_layers)) return e;
    if (!tg_frame_supported((int)f->width, (int)f->height, (int)f->tile_w, (int)f->tile_h)) {
        set_error("%s: more than 256 tile columns or rows", fn);
        return TG_E_ARG;
    }
    return 0;
}

// Zeroes the gradients, 16 bytes a thread.
__global__ __launch_bounds__(256) void zero_gradients_kernel(real4 *p, int64_t n4) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n4) p[i] = make_real4(0.0f, 0.0f, 0.0f, 0.0f);
}

static OrderStore frame_order(const tg_frame &f, const FrameLayout &L, char *kept) {
    if (f.flags & TG_FRAME_ORDER_PLANES) return OrderStore{(uint16_t *)(kept + L.order), f.max_layers * f.width * f.height, 0};
    if (f.flags & TG_FRAME_ORDER_POOL) {
        const int pixels = order_pool_pixels((int)f.tile_w, (int)f.tile_h);
        return OrderStore{(uint16_t *)(kept + L.order), f.n_triangles > kShortList ? f.key_capacity * pixels : 0, pixels};
    }
    return OrderStore{nullptr, 0, 0};
}
#endif

}  // namespace tg

using namespace tg;

extern "C" int tg_frame_supported(int width, int height, int tile_w, int tile_h) {
    if (!tg_bin_frame_supported(width, height, tile_w, tile_h)) return 0;
    return frame_grid_fits(ceil_div(width, tile_w), ceil_div(height, tile_h)) ? 1 : 0;
}

#ifdef TG_DOUBLE_PRECISION
static int no_frame(const char *fn) {
    set_error("%s: float build only", fn);
    return TG_E_ARG;
}
extern "C" int tg_frame_layout(const tg_frame *, int64_t *) { return no_frame("tg_frame_layout"); }
extern "C" int tg_frame_has_records(const tg_frame *) { return 0; }
extern "C" int tg_frame_forward(tg_frame *) { return no_frame("tg_frame_forward"); }
extern "C" int tg_frame_backward(const tg_frame *) { return no_frame("tg_frame_backward"); }
#else
extern "C" int tg_frame_has_records(const tg_frame *f) { return check_frame("tg_frame_has_records", f) == 0 && has_records(*f); }

extern "C" int tg_frame_layout(const tg_frame *f, int64_t *out) {
    if (int e = check_frame("tg_frame_layout", f)) return e;
    if (!out) { set_error("tg_frame_layout: null pointer"); return TG_E_ARG; }
    const FrameLayout L = frame_layout(*f);
    const int64_t words[TG_FRAME_LAYOUT_WORDS] = {
        (int64_t)L.kept_bytes, (int64_t)L.scratch_bytes,
        (int64_t)tg_bin_frame_workspace_bytes((int32_t)f->n_triangles, f->key_capacity, (int)f->width, (int)f->height, (int)f->tile_w, (int)f->tile_h),
        (int64_t)L.status, (int64_t)L.ids, (int64_t)L.offsets, (int64_t)L.bary, (int64_t)L.weights, (int64_t)L.ends, (int64_t)L.last,
        (int64_t)L.last_depth, (int64_t)L.order, (int64_t)L.masks};
    for (int i = 0; i < TG_FRAME_LAYOUT_WORDS; i++) out[i] = words[i];
    return 0;
}

extern "C" int tg_frame_forward(tg_frame *f) {
    if (int e = check_frame("tg_frame_forward", f)) return e;
    const FrameLayout L = frame_layout(*f);
    if (f->kept_bytes < (int64_t)L.kept_bytes || f->scratch_bytes < (int64_t)L.scratch_bytes) {
        set_error("tg_frame_forward: buffers of %lld and %lld bytes, need %zu and %zu", (long long)f->kept_bytes,
                  (long long)f->scratch_bytes, L.kept_bytes, L.scratch_bytes);
        return TG_E_WORKSPACE;
    }
    if (!f->kept || !f->scratch || !f->host || !f->frame || (f->frame_bytes & 7) || ((uintptr_t)f->kept & 255) || ((uintptr_t)f->scratch & 255) || ((uintptr_t)f->host & 7)) {
        set_error("tg_frame_forward: null or misaligned buffer");
        return TG_E_ARG;
    }
    char *kept = (char *)f->kept, *scratch = (char *)f->scratch;
    const int W = (int)f->width, H = (int)f->height, tw = (int)f->tile_w, th = (int)f->tile_h;
    const int tiles_x = ceil_div(W, tw), tiles_y = ceil_div(H, th), tiles = tiles_x * tiles_y;
    const int32_t V = (int32_t)f->n_vertices, M = (int32_t)f->n_triangles;
    uint32_t *status = (uint32_t *)(kept + L.status);
    uint32_t *total_and_status = (uint32_t *)((char *)f->frame + f->frame_bytes);
    uint64_t *keys = (uint64_t *)(scratch + L.keys);
    uint32_t *ids = (uint32_t *)(kept + L.ids);
    int32_t *offsets = (int32_t *)(kept + L.offsets);
    real *bary = (real *)(kept + L.bary);
    real4 *records = has_records(*f) ? (real4 *)bary : nullptr;
    volatile uint32_t *host = f->host;
    const int64_t longest = f->key_capacity < f->n_triangles ? f->key_capacity : f->n_triangles;  // a triangle is in a list once
    LongTiles long_tiles;
    if (L.long_limit)
        long_tiles = LongTiles{(int32_t *)(scratch + L.long_tiles) + kLongTileCounters, (int32_t *)(scratch + L.all_long_tiles), L.long_limit,
                               std::min<int64_t>(tiles, f->key_capacity / L.long_limit), (uint32_t *)(scratch + L.long_tiles)};
    if (f->phases & TG_FRAME_BIN) {
        host[1] = 0;
        host[2] = TG_FRAME_PENDING;
        if (int e = bin_frame(f->vertices, V, f->indices, M, W, H, tw, th, keys, ids, f->key_capacity, total_and_status, f->frame,
                              (size_t)f->frame_bytes, (uint32_t)f->epoch, scratch + L.sort, L.zero_bytes, status, bary,
                              (uint64_t *)f->host, f->stream, f->colors, f->opacities, records))
            return e;
    }
    if (f->phases & TG_FRAME_LISTS) {
        int in_alt = 0;  // two passes: the pairs are back where they started
        if (int e = build_frame_lists(f->frame, (uint32_t)f->epoch, f->key_capacity, total_and_status, longest, tiles_x, tiles_y, keys,
                                      ids, (uint64_t *)(scratch + L.keys_alt), (uint32_t *)(scratch + L.values_alt), offsets,
                                      scratch + L.sort, L.sort_bytes, status, &in_alt, long_tiles, f->stream))
            return e;
    }
    if (f->phases & TG_FRAME_RASTER) {
        real *bounds = nullptr;
        int32_t *far_start = nullptr;
        if (f->flags & TG_FRAME_LIST_BOUNDS) {
            bounds = (real *)(scratch + L.bounds);
            far_start = (int32_t *)(scratch + L.far_start);
            if (int e = tg_list_bounds(f->vertices, V, f->indices, M, keys, (const int32_t *)ids, offsets, tiles,
                                       (real *)(scratch + L.low), bounds, far_start, f->stream))
                return e;
        }
        const bool backward = f->flags & TG_FRAME_BACKWARD;
        if (int e = render_forward(f->vertices, f->indices, f->colors, f->opacities, (const int32_t *)ids, offsets, bary, W, H, tw, th,
                                   (real)f->early_stopping_threshold, (int)f->per_pixel_sort, (int)f->max_layers, f->image, f->depthmap,
                                   (real *)(kept + L.weights), (int32_t *)(kept + L.ends), backward ? (int32_t *)(kept + L.last) : nullptr,
                                   backward && f->per_pixel_sort ? (real *)(kept + L.last_depth) : nullptr, frame_order(*f, L, kept),
                                   (f->flags & TG_FRAME_HIT_MASKS) ? (uint64_t *)(kept + L.masks) : nullptr, bounds, far_start, status,
                                   (uint32_t *)f->host + 2, longest, long_tiles, records, f->stream))
            return e;
    }
    if (f->phases & TG_FRAME_WAIT) {
        if (int e = tg_frame_wait(f->host, 1, 0, f->stream)) return e;
        f->n_keys = host[0];
        f->counted = host[1];
    }
    return 0;
}

extern "C" int tg_frame_backward(const tg_frame *f) {
    if (int e = check_frame("tg_frame_backward", f)) return e;
    const FrameLayout L = frame_layout(*f);
    if (!f->kept || f->kept_bytes < (int64_t)L.kept_bytes || !(f->flags & TG_FRAME_BACKWARD) || !f->gradients ||
        ((uintptr_t)f->gradients & 15) || ((uintptr_t)f->kept & 255) || (f->per_pixel_sort && (!f->block || ((uintptr_t)f->block & 15)))) {
        set_error("tg_frame_backward: null, small or misaligned buffer, or a frame rendered without TG_FRAME_BACKWARD");
        return TG_E_ARG;
    }
    const int64_t given = f->phases >> 16;  // blocks
    const bool by_count = f->phases & TG_FRAME_GRADIENT_COPIES;
    const int copies = by_count ? (int)given : f->per_pixel_sort ? 1 : 0;
    if ((by_count && given != 0 && given != 1 && given != 8) || (copies && (!f->block || ((uintptr_t)f->block & 15)))) {
        set_error("tg_frame_backward: null or misaligned block, or a number of blocks that is not 0, 1 or 8");
        return TG_E_ARG;
    }
    char *kept = (char *)f->kept;
    const int64_t V = f->n_vertices;
    if (V == 0) return 0;
    // One zero fill for the three gradients.  Where there are many vertices, or many waves meet in one, the eight gradients of a vertex lie
    // in a 32-byte sector of a (V,8) block while the kernel runs, and the three arrays are copied out afterwards: the atomics of a run
    // then fall into three sectors and not nine.  The copy is another launch, and sums of few vertices stay in the L2 whatever their
    // places, so not for the smallest images, and in tile order, with less than half the atomics, only where triangles share vertices or
    // vertices are many and the image is large.  Kernels, us, dense and by the block with the copy.  Tile order, a soup of 3 * 10^6 vertices 577, 360 + 28,
    // 3 * 10^5 82, 68 + 6, 9 * 10^4 36.2, 31.7 + 4.8, 5 * 10^4 with a heavy tail 375, 319 + 5, 3 * 10^4 18.8, 18.4 + 2.9; a mesh of
    // 650 000 on 1920 x 1080 440, 310 + 8, 28 000 on 1235 x 981 91, 62 + 5, 1200 there 124, 58 + 5, 5000 on 500 x 400 26, 23 + 2.4,
    // on 256 x 256 24.4, 22.4 + 2.4.  Per-pixel order, a soup of 9 * 10^4 43.8, 36.3 + 4.7, of 1500 with a heavy tail on 256 x 256
    // 98, 92.5 + 4.6, 300 on 128 x 128 38.9, 35.3 + 3.5, 60 on 50 x 50 10.2, 10.1 + 1.4; a mesh of 1200 on 1235 x 981 137, 67 + 5.
    // A sector that several XCDs add to goes from L2 to L2, and triangles that cover hundreds of tiles are in all of them.  So each XCD
    // has a block of its own where triangles are in 20 waves on average, a tile counted as all of its waves (with more vertices than 131072,
    // or than a quarter of the pixels, the zeros and the copy, 512 bytes a vertex, cost what it gains).  Whole frames, us, one block and eight: heavy tails on 1100 x 1000 to 1230 x 1080, 1291
    // triangles in per-pixel order 381, 213, 15 800 617, 481, 30 000 728, 514, 2072 in tile order 400, 204, 15 800 436, 296; no
    // heavy tail, 20 000 large ones 988, 989, 3000 on 1024 x 1024 130, 131.  Below the line: 60 000 with a heavy tail 550, 563,
    // 33 331 in tiles of 8 x 8 273, 278, a mesh of 20 000 124, 127.  The backward pass alone near it, all of one size: 20 000 on
    // 1024 x 1024, 15 waves a triangle 63, 71, 21 waves 93, 102; 1000 there, 16 waves 22, 24, 300 on 256 x 256, 20 waves 19.3, 21.4; in tile order
    // 75, 84 (21 waves), 15.6, 19.2 (20); with a heavy tail, which their mean does not tell, 1500 on 256 x 256, 25 waves 66, 64 and 40, 35.
    real *sums = copies ? f->block : f->gradients;
    const int64_t n4 = 2 * V * max(copies, 1);
    TG_LAUNCH(zero_gradients_kernel, dim3((unsigned)ceil_div64(n4, 256)), dim3(256), 0, (hipStream_t)f->stream, (real4 *)sums, n4);
    if (int e = check_launch("zero_gradients_kernel")) return e;
    const int stride = copies ? 8 : 0;
    if (int e = render_backward(f->grad_image, f->grad_depthmap, f->vertices, f->indices, f->colors, f->opacities,
                                (const int32_t *)(kept + L.ids), (const int32_t *)(kept + L.offsets), (const real *)(kept + L.bary), f->image,
                                f->depthmap, (const real *)(kept + L.weights), (const int32_t *)(kept + L.ends),
                                (const int32_t *)(kept + L.last), f->per_pixel_sort ? (const real *)(kept + L.last_depth) : nullptr,
                                frame_order(*f, L, kept), (f->flags & TG_FRAME_HIT_MASKS) ? (const uint64_t *)(kept + L.masks) : nullptr,
                                (int)f->width, (int)f->height, (int)f->tile_w, (int)f->tile_h, (real)f->early_stopping_threshold,
                                (int)f->per_pixel_sort, (int)f->max_layers, sums, stride ? sums + 4 : sums + 4 * V,
                                stride ? sums + 7 : sums + 7 * V, stride ? stride : 4, stride ? stride : 3, stride ? stride : 1, copies > 1 ? 8 * V : 0,
                                (const uint32_t *)(kept + L.status), f->key_capacity, has_records(*f) ? (const real4 *)(kept + L.bary) : nullptr, f->stream))
        return e;
    if (!copies) return 0;
    return split_gradient_block(f->block, V, copies, f->gradients, f->gradients + 4 * V, f->gradients + 7 * V, f->stream);
}
#endif

extern "C" int tg_frame_gradient_copies(const tg_frame *f) { return f ? gradient_copies(*f) : 0; }

extern "C" int tg_frame_wait(const uint32_t *host, int word, uint32_t pending, void *stream) {
    if (!host || word < 0 || word > 3) {
        set_error("tg_frame_wait: null pointer or no such word");
        return TG_E_ARG;
    }
    const volatile uint32_t *at = host + word;
    // the word is written early in a kernel; looking for it costs neither an event nor the wake-up of a sleeping thread.
    // A stream busy with something long, or a frame whose kernels failed, ends the looking and waits for the stream.
    const auto start = std::chrono::steady_clock::now();
    for (int looks = 0; *at == pending; looks++) {
        _mm_pause();
        if ((looks & 63) == 63 && std::chrono::steady_clock::now() - start > std::chrono::milliseconds(50)) {
            const hipError_t e = hipStreamSynchronize((hipStream_t)stream);
            if (e != hipSuccess) {
                set_error("tg_frame_wait: %s", hipGetErrorString(e));
                return (int)e;
            }
            if (*at != pending) break;
            set_error("tg_frame_wait: the stream is done and the word is not there");
            return TG_E_ARG;
        }
    }
    std::atomic_thread_fence(std::memory_order_acquire);
    return 0;
}
