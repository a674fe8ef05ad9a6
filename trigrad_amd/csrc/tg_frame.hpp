// tg_frame.hpp -- the stages of a frame as the one-call route (tg_frame.hip) strings them together: nothing below needs
// the number of keys K on the host.
#pragma once
#include "tg_raster.hpp"

namespace tg {

// A number of pairs that is known on the device only: `word` points at tg_bin_frame's pair (K, epoch of an expired wait),
// `capacity` is what the buffers hold.  With a null `word` the number is the one the host passed.  No pairs, so empty lists,
// where the host runs the frame again: more keys than the buffers hold, or a wait of the scan that expired, whose K is the
// sum of what it had and does not belong to the digit totals that the sort's bases are made from.
struct FrameCount {
    const uint32_t *word = nullptr;
    uint32_t capacity = 0, epoch = 0;
    __host__ __device__ __forceinline__ bool expired() const { return word && word[1] == epoch; }
    __host__ __device__ __forceinline__ int64_t pairs(int64_t given) const {
        if (!word) return given;
        const uint32_t n = word[0];
        return !expired() && n <= capacity ? n : 0;
    }
};

// The tiles with the longest lists, for a kernel that starts with them, or shares their work out: a tile's list is one
// workgroup's serial work, and what the whole launch waits for is the longest.  The segment sort, which makes the lists'
// bounds, notes every tile with `limit` entries or more.  words: how many there are, then the first kLongTileSlots of them; all:
// all of them; most: no more of them are possible.  Null words: there can be none.
constexpr int kLongTileSlots = 128, kLongTileCounters = 4;
struct LongTiles {
    int32_t *words = nullptr;
    int32_t *all = nullptr;  // room for every tile
    int limit = 0;
    int64_t most = 0;
    uint32_t *taken = nullptr;  // a counter for each of a tile's workgroups, for a launch that shares the work out; zero between launches
};

// tg_bin_frame with outputs more: the bary matrices, or (records) the triangles' records in their place, and K for the host; all may be null.
int bin_frame(const real *vertices, int32_t n_vertices, const int32_t *indices, int32_t n_triangles, int width, int height, int tile_w,
              int tile_h, uint64_t *keys, uint32_t *values, int64_t key_capacity, uint32_t *total_and_status, void *frame,
              size_t frame_bytes, uint32_t epoch, void *zero, size_t zero_bytes, uint32_t *clear_word, real *bary, uint64_t *host_total,
              void *stream, const real *colors, const real *opacities, real4 *records);
int build_frame_lists(void *frame, uint32_t epoch, int64_t n_keys, const uint32_t *total_and_status, int64_t longest, int tiles_x,
                      int tiles_y, uint64_t *keys, uint32_t *values, uint64_t *keys_alt, uint32_t *values_alt, int32_t *offsets,
                      void *workspace, size_t workspace_bytes, uint32_t *status, int *result_in_alt, const LongTiles &long_tiles,
                      void *stream);
// records: the triangles' records, or null.
// host_status: receives the list kernels' status word, in memory the host reads; longest: no list holds more entries.
int render_forward(const real *vertices, const int32_t *indices, const real *colors, const real *opacities, const int32_t *sorted_ids,
                   const int32_t *offsets, const real *bary, int width, int height, int tile_w, int tile_h, real early_stopping_threshold,
                   int per_pixel_sort, int max_layers, real *image, real *depthmap, real *final_weights, int32_t *ends, int32_t *last,
                   real *last_depth, const OrderStore &order, uint64_t *hit_masks, const real *batch_bounds, const int32_t *far_start,
                   const uint32_t *list_status, uint32_t *host_status, int64_t longest, const LongTiles &long_tiles, const real4 *records, void *stream);
int render_backward(const real *grad_image, const real *grad_depthmap, const real *vertices, const int32_t *indices, const real *colors,
                    const real *opacities, const int32_t *sorted_ids, const int32_t *offsets, const real *bary, const real *image,
                    const real *depthmap, const real *final_weights, const int32_t *ends, const int32_t *last, const real *last_depth,
                    const OrderStore &order, const uint64_t *hit_masks, int width, int height, int tile_w, int tile_h,
                    real early_stopping_threshold, int per_pixel_sort, int max_layers, real *grad_vertices, real *grad_colors,
                    real *grad_opacities, int vertex_stride, int color_stride, int opacity_stride, int64_t copy_stride,
                    const uint32_t *list_status, int64_t n_keys, const real4 *records, void *stream);  // n_keys: about how many, for what does not have to be right; 0 if it is not known
// The three arrays out of `copies` (V,8) blocks behind each other: their sum.
int split_gradient_block(const real *block, int64_t n_vertices, int copies, real *grad_vertices, real *grad_colors, real *grad_opacities, void *stream);
bool frame_grid_fits(int tiles_x, int tiles_y);  // at most 256 tile columns and rows: the sort passes are the tile's coordinates

}  // namespace tg
