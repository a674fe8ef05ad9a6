// tg_forward.hpp -- what the forward kernels share: their outputs, which tile a workgroup takes, and the tile-order pass of one
// tile.
#pragma once
#include "tg_frame.hpp"
#include "tg_raster.hpp"

namespace tg {

struct ForwardOut {
    real4 *image;
    real *depthmap;
    real *weights;
    int32_t *ends;
    int32_t *last;
    real *last_depth;
    OrderStore order;    // blend order: list positions relative to the tile's start
    uint64_t *hit_masks; // tile order: which list entries cover which pixel, 64 entries per word (see hit_mask_chunk); may be null
    const uint32_t *list_status;  // status word of the kernels that made the lists (TG_STATUS_*); may be null
    uint32_t *host_status;        // where the host looks for that word (memory of its own); may be null
    LongTiles long_tiles;
    int long_rows;                // rows of workgroups at the start of the grid, for the long tiles
};

// The workgroups in the first long_rows rows of a forward launch take the tiles with the longest lists (LongTiles), the others
// the rest in the order of tile_of_workgroup.  A frame without a long tile loses 1 us by the workgroups that find none.
__device__ __forceinline__ int long_group(const ForwardOut &o) { return (int)(blockIdx.y * gridDim.x + blockIdx.x); }
__device__ __forceinline__ int long_groups(const ForwardOut &o) { return o.long_rows * (int)gridDim.x; }
__device__ __forceinline__ TileId tile_of_index(int index) {
    TileId t;
    int columns = (int)gridDim.x;
    asm volatile("" : "+s"(columns));  // the division's constants are made here, not kept in registers by the loop around the call
    t.index = index;
    t.y = index / columns;
    t.x = index - t.y * columns;
    return t;
}
// A launch that shares the long tiles' work out takes them all; one that only starts with them takes the first few, whole.
__device__ __forceinline__ bool is_long_tile(const ForwardOut &o, int n_entries) { return o.long_rows && n_entries >= o.long_tiles.limit; }
__device__ __forceinline__ int tiles_started_first(const ForwardOut &o) { return min(min(o.long_tiles.words[0], kLongTileSlots), long_groups(o)); }
__device__ __forceinline__ bool is_started_first(const ForwardOut &o, int tile, int n_entries) {
    if (!is_long_tile(o, n_entries)) return false;
    const int n = tiles_started_first(o), lane = threadIdx.x & (kWave - 1);
    bool found = false;
    for (int slot = lane; slot < n; slot += kWave) found = found || o.long_tiles.words[1 + slot] == tile;
    return __builtin_amdgcn_ballot_w64(found) != 0;
}

// Lists whose sort gave up a wait are not to be read (unwritten entries may name anything): the frame's pixels
// are marked instead, so that the caller sees it in the image itself.
__device__ __forceinline__ bool lists_invalid(const ForwardOut &o) {
    if (!o.list_status) return false;
    const uint32_t status = *o.list_status;
    if (o.host_status && (blockIdx.x | blockIdx.y | blockIdx.z | threadIdx.x) == 0)
        __hip_atomic_store(o.host_status, status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    return status != TG_STATUS_OK;
}
__device__ __forceinline__ void mark_tile_invalid(const RasterArgs &a, const ForwardOut &o) {
    if ((int)blockIdx.y < o.long_rows) return;
    const PixelCoord p = pixel_of_thread(a, tile_of_workgroup<kTileBandForward, kChunkForward>(o.long_rows));
    if (!p.valid) return;
    const real nan = std::numeric_limits<real>::quiet_NaN();
    o.image[p.index] = make_real4(nan, nan, nan, nan);
    o.depthmap[p.index] = nan;
    o.weights[p.index] = 0.0f;
    o.ends[p.index] = 0;
    if (o.last) o.last[p.index] = 0;
    if (o.last_depth) o.last_depth[p.index] = nan;
}

__device__ __forceinline__ void write_pixel(const ForwardOut &o, const PixelCoord &p, PixelState s, int last, real last_depth) {
    // render.cu:609-618
    real depth;
    if (s.weight > kEffZero) {
        depth = s.depth / s.weight;
    } else {
        depth = __builtin_inff();
        s.weight = 0.0f;
    }
    o.depthmap[p.index] = depth;
    o.weights[p.index] = s.weight;
    o.ends[p.index] = s.blended;
    if (o.last) o.last[p.index] = last;
    if (o.last_depth) o.last_depth[p.index] = last_depth;
    o.image[p.index] = make_real4(s.c0, s.c1, s.c2, s.alpha);
}

// The tile-order forward pass of one tile, a pixel per thread.
struct TileOrderLds {
    BlendRecord rec[kBatch];
    uint8_t touch[kBatch];
    WaveRect rects[kMaxTileWaves];
    int last;
};
template <bool kPacked>
__device__ __forceinline__ void tile_order_tile(const RasterArgs &a, const ForwardOut &out, const TileId &tile_id, int start, int end, TileOrderLds &lds) {
    BlendRecord *s_rec = lds.rec;
    uint8_t *s_touch = lds.touch;
    WaveRect *s_rects = lds.rects;
    const int tid = threadIdx.x;
    const int wave = tid / kWave;
    const int n_waves = blockDim.x / kWave;
    const int tile = tile_id.index;
    const PixelCoord p = pixel_of_thread(a, tile_id);
    publish_wave_rect(a, p, s_rects);
    const bool tests_small = tests_small_entries(a, end - start, (int)(gridDim.x * (gridDim.y - out.long_rows)));
    uint64_t *const masks = out.hit_masks ? out.hit_masks + hit_mask_head_words(out.long_rows) : nullptr;

    PixelState s;
    int last = 0;
    for (int batch = start; batch < end; batch += kBatch) {
        const bool running = p.valid && s.alpha > a.thr && s.blended < a.max_layers;
        if (!__syncthreads_or(running)) break;
        const int nb = min(kBatch, end - batch);
        for (int e = tid; e < nb; e += blockDim.x) {
            gather_blend<kPacked, true>(a, batch + e, s_rec[e]);
            s_touch[e] = (uint8_t)(waves_touched(s_rec[e].m, s_rects, n_waves) | small_entry(a, s_rec[e].extent, tests_small));
        }
        __syncthreads();
        // 1. inside tests; a lane keeps its hits as a 256-bit mask
        uint64_t m[kBatch / kWave];
        batch_hit_mask<kBatch / kWave>(s_rec, s_touch, s_rects, nb, wave, p.px, p.py, m);
        if (!running) {
#pragma unroll
            for (int wd = 0; wd < kBatch / kWave; wd++) m[wd] = 0;
        }
        if (masks) {
            // kept for the backward pass, which then has no inside test to repeat
            const int64_t chunk = hit_mask_chunk(start, tile, batch - start);
            const int64_t slots = (int64_t)gridDim.z * blockDim.x, slot = (int64_t)blockIdx.z * blockDim.x + tid;
#pragma unroll
            for (int wd = 0; wd < kBatch / kWave; wd++)
                if (wd * kWave < nb) masks[(chunk + wd) * slots + slot] = m[wd];
        }
        // 2. every lane composites its own hits in list order, so the blend arithmetic
        //    runs with as many lanes busy as there are pixels with a fragment left
        while (true) {
            int e = -1;
            if (s.alpha > a.thr && s.blended < a.max_layers) e = pop_lowest<kBatch / kWave>(m);  // render.cu:578, tested before every fragment
            if (__builtin_amdgcn_ballot_w64(e >= 0) == 0) break;  // wave-uniform
            if (e >= 0) {
                const BlendRecord &r = s_rec[e];
                real b0, b1, b2;
                bary_apply(r.m, p.px, p.py, b0, b1, b2);
                blend_fragment(s, r, b0, b1, b2);
                last = batch + e - start + 1;
            }
        }
    }
    if (p.valid) write_pixel(out, p, s, last, 0.0f);
    if (out.hit_masks) {
        // how far into the list this workgroup's pixels got
        int &s_last = lds.last;
        __syncthreads();
        if (tid == 0) s_last = 0;
        __syncthreads();
        int wave_last = p.valid ? last : 0;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) wave_last = max(wave_last, __shfl_xor(wave_last, off, kWave));
        if ((tid & (kWave - 1)) == 0 && wave_last > 0) atomicMax(&s_last, wave_last);
        __syncthreads();
        if (tid == 0) out.hit_masks[hit_mask_head_index(tile)] = (uint64_t)s_last;
    }
}

// Eight waves per SIMD (63 registers, nothing in scratch memory): 212 -> 194 us against the 73 registers it would take
// (10^6 triangles, 1920 x 1080).  No bound in double precision: held to the five waves that the LDS allows it spills (8 x 8
// tiles: 112 -> 123 us).  The tiles with the longest lists are started first, as far as there are workgroups for them; a launch
// of few workgroups shares their work out instead (forward_tile_order_few_kernel).
template <bool kPacked>
__global__ __launch_bounds__(kTileThreads, sizeof(real) == 4 ? 8 : 1) void forward_tile_order_kernel(RasterArgs a, ForwardOut out) {
    __shared__ TileOrderLds s;
    if (lists_invalid(out)) {  // the same for the whole launch
        mark_tile_invalid(a, out);
        return;
    }
    const bool first = (int)blockIdx.y < out.long_rows;
    if (first && long_group(out) >= tiles_started_first(out)) return;
    const TileId tile = first ? tile_of_index(out.long_tiles.words[1 + long_group(out)]) : tile_of_workgroup<kTileBandForward, kChunkForward>(out.long_rows);
    const int start = a.offsets[tile.index], end = a.offsets[tile.index + 1];
    if (!first && is_started_first(out, tile.index, end - start)) return;
    tile_order_tile<kPacked>(a, out, tile, start, end, s);
}

// The kernels of launches with few workgroups (tg_forward_few.hip): forward_tile_order_kernel's, and forward_pixel_order_kernel
// with all of a candidate list's places in LDS, and where the tiles' workgroups help with the long tiles.  Null in the double
// build, which has none of them: every launch has all places in LDS there, and long tiles are noted by tg_frame_forward, a call of
// the float build.
constexpr int kFewTileGroups = 1024;
constexpr bool kSharesLongTiles = sizeof(real) == 4;
using ForwardKernel = void (*)(RasterArgs, ForwardOut);
ForwardKernel tile_order_few_kernel();
ForwardKernel pixel_order_few_kernel(bool in_turn);
ForwardKernel pixel_order_helping_kernel(bool all_places);

// The instances that read triangles' records (tg_forward_packed.hip).  Null in the double build.
using LongListsKernel = void (*)(RasterArgs, ForwardOut, int, int);
ForwardKernel packed_tile_order_kernel();
ForwardKernel packed_tile_order_few_kernel();
ForwardKernel packed_pixel_order_kernel(bool tiles_help, bool all_places, bool in_turn);
ForwardKernel packed_pixel_order_bounds_kernel(bool in_turn);
LongListsKernel packed_pixel_order_long_lists_kernel();

}  // namespace tg
