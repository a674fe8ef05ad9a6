// tg_forward_few.hpp -- the forward kernels of launches with few workgroups: in tile order one that shares the long tiles' work
// out, in per-pixel order one whose workgroups help with the long tiles.  (float build)
#pragma once
#include "tg_forward_pixel.hpp"

namespace tg {

// A wave's share (64 pixels; the part-th of its workgroup's) of a tile with a long list, by the four waves of a workgroup, in
// tile order: each tests 64 of 256 entries, lane = entry, from registers; the records of those that are hit go to LDS, and the
// first wave composites them in list order.  500 000 triangles of a mesh, 500 x 500 (longest list 5500, a tile one workgroup's
// chain before): 367 -> 127 us.  s_hits: per wave, which of its 64 entries cover a pixel, then which of them cover any, then which
// of those are staged.
template <bool kPacked>
__device__ __forceinline__ void long_tile_part(const RasterArgs &a, const ForwardOut &out, const TileId &tile, int part, BlendRecord *s_rec,
                                               uint64_t (*s_hits)[kWave + 2]) {
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));  // what depends on it is made here, not kept in registers by the loop around the call
    const int lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int start = a.offsets[tile.index], end = a.offsets[tile.index + 1];
    const int slot = (blockIdx.z * kMaxTileWaves + part) * kWave + lane;
    const PixelCoord p = pixel_of_slot(a, tile.x, tile.y, slot);
    const WaveRect rect = wave_rect(a, p);
    const bool squares = ((a.tw | a.th) & 7) == 0;
    PixelState s;  // of the first wave
    int last = 0;
    // an entry's matrix and vertex numbers are asked for while the entries before it are composited, its triangle's number
    // before that; what only the entries that are hit need is read when it is known which they are
    std::conditional_t<kPacked, PackedParts, DepthParts> next;
    const auto entry = [&](int first) { return min(first + tid, end - 1); };
    next.fetch_triangle(a, entry(start));
    int fetched = next.tri;  // the triangle whose matrix it is
    next.fetch_matrix(a);
    next.fetch_triangle(a, entry(start + kTileThreads));
    for (int first = start; first < end; first += kTileThreads) {
        const bool running = wave == 0 && p.valid && s.alpha > a.thr && s.blended < a.max_layers;
        if (!__syncthreads_or(running)) break;
        real matrix[9];
        next.get_matrix(matrix);
        [[maybe_unused]] int3v id;
        [[maybe_unused]] const int tri = fetched;
        if constexpr (!kPacked) id = next.id;
        fetched = next.tri;
        next.fetch_matrix(a);
        next.fetch_triangle(a, entry(first + 2 * kTileThreads));
        uint64_t hit;
        const uint64_t m = wave_hits(matrix, first + tid < end, squares, rect, p.px, p.py, hit);
        s_hits[wave][lane] = m;
        if (lane == 0) s_hits[wave][kWave] = hit;
        if (out.hit_masks && first + wave * kWave < end) {
            const int64_t chunk = hit_mask_chunk(start, tile.index, first + wave * kWave - start);
            out.hit_masks[hit_mask_head_words(out.long_rows) + chunk * ((int64_t)gridDim.z * kTileThreads) + slot] = m;
        }
        __syncthreads();
        int before = 0, total = 0;
#pragma unroll
        for (int w = 0; w < kMaxTileWaves; w++) {
            const int count = __builtin_popcountll(s_hits[w][kWave]);
            if (w < wave) before += count;
            total += count;
        }
        const int rank = before + (int)lanes_below_mask(hit);
        for (int round = 0; round < total; round += kBatch) {  // the same for the workgroup
            const bool staged = ((hit >> lane) & 1) && rank >= round && rank < round + kBatch;
            const uint64_t group = __builtin_amdgcn_ballot_w64(staged);
            if (lane == 0) s_hits[wave][kWave + 1] = group;
            if constexpr (kPacked) {
                if (staged) gather_record(a, matrix, tri, s_rec[rank - round]);
            } else {
                if (staged) gather_record(a, matrix, id, s_rec[rank - round]);
            }
            __syncthreads();
            if (wave == 0) {
                int base = 0;
                for (int w = 0; w < kMaxTileWaves; w++) {
                    const uint64_t there = s_hits[w][kWave + 1];
                    uint64_t bits = s_hits[w][lane] & there;
                    while (true) {
                        const bool more = bits && p.valid && s.alpha > a.thr && s.blended < a.max_layers;  // render.cu:578, tested before every fragment
                        if (__builtin_amdgcn_ballot_w64(more) == 0) break;  // wave-uniform
                        if (!more) continue;
                        const int e = __builtin_ctzll(bits);
                        bits &= bits - 1;
                        const BlendRecord &b = s_rec[base + __builtin_popcountll(there & ((1ull << e) - 1))];
                        real b0, b1, b2;
                        bary_apply(b.m, p.px, p.py, b0, b1, b2);
                        blend_fragment(s, b, b0, b1, b2);
                        last = first - start + w * kWave + e + 1;
                    }
                    base += __builtin_popcountll(there);
                }
            }
            __syncthreads();
        }
    }
    if (wave == 0 && p.valid) write_pixel(out, p, s, last, 0.0f);
    // the tile's pixels are four workgroups': the backward pass finds out for itself how far they got
    if (out.hit_masks && tid == 0) out.hit_masks[hit_mask_head_index(tile.index)] = ~0ull;
}

// Shared out, a tile with a long list is four waves' work for each of its squares.  That takes 120 registers, four waves per
// SIMD, which up to 1024 workgroups do not need more of; a launch of more is better off with eight (forward_tile_order_kernel).
template <bool kPacked>
__global__ __launch_bounds__(kTileThreads, 4) void forward_tile_order_few_kernel(RasterArgs a, ForwardOut out) {
    __shared__ TileOrderLds s;
    if (lists_invalid(out)) {  // the same for the whole launch
        mark_tile_invalid(a, out);
        return;
    }
    if ((int)blockIdx.y < out.long_rows) {
        __shared__ uint64_t s_hits[kMaxTileWaves][kWave + 2];
        const int n_items = kMaxTileWaves * out.long_tiles.words[0];
        for (int item = long_group(out); item < n_items; item += long_groups(out))
            long_tile_part<kPacked>(a, out, tile_of_index(out.long_tiles.all[item / kMaxTileWaves]), item % kMaxTileWaves, s.rec, s_hits);
        return;
    }
    const TileId tile = tile_of_workgroup<kTileBandForward, kChunkForward>(out.long_rows);
    const int start = a.offsets[tile.index], end = a.offsets[tile.index + 1];
    if (is_long_tile(out, end - start)) return;
    tile_order_tile<kPacked>(a, out, tile, start, end, s);
}

// forward_pixel_order_kernel with 16-bit positions of a launch whose workgroups run at once: those that are done with a tile's list help with the long tiles.
// So there need not be a workgroup in front of the others for each item (a long tile's square) that there may be, and there had
// better not: they change which tiles meet on a CU, which a launch of one generation has no others to make up for (20 000 large
// triangles on 1024 tiles without a limit on the layers, forward, us: 128 in front 366, 1024 387), and 128 alone find too much
// (1024 tiles, 200 with 3000 large faint triangles, frames, us: 128 1735, 1024 772, 128 and the tiles' 793; 100 such tiles 970, 573,
// 603; 784 tiles, 30 such 310, 310, 310).
//
// The first items are those of the workgroups in front, in order.  If there are more, every workgroup that is done draws the next
// one until it draws one beyond the last: a draw for each item behind the first ones, and one more of every workgroup.  That is one
// for each item and each tile in all; the last of them finds the counter at items + tiles - 1 and leaves it at zero, for another
// launch.
static_assert(kMaxTilePixels <= kLongTileCounters * kTileThreads, "a counter for each of a tile's workgroups");
template <int kHead, bool kPacked>
__global__ __launch_bounds__(kTileThreads, short_list_waves(kHead)) void forward_pixel_order_helping_kernel(RasterArgs a, ForwardOut out) {
    extern __shared__ __align__(16) unsigned char s_dyn[];
    __shared__ uint8_t s_touch[kSelectBatchShort];
    __shared__ WaveRect s_rects[kMaxTileWaves];
    __shared__ int s_drawn;
    if (lists_invalid(out)) {  // the same for the whole launch
        mark_tile_invalid(a, out);
        return;
    }
    const bool first = (int)blockIdx.y < out.long_rows;
    if (!first) {
        const TileId tile = tile_of_workgroup<kTileBandForward, kChunkForward>(out.long_rows);
        const int n = a.offsets[tile.index + 1] - a.offsets[tile.index];
        if (!is_long_tile(out, n) && n <= kShortList)
            pixel_order_tile<kSelectBatchShort, uint16_t, true, kHead, kPacked>(a, out, tile.x, tile.y, gridDim.x, gridDim.x * (gridDim.y - out.long_rows), s_dyn, s_touch, s_rects);
    }
    const auto items = [&] { return kMaxTileWaves * out.long_tiles.words[0]; };
    const auto draw = [&] {
        if (items() <= long_groups(out)) return items();
        __syncthreads();  // all have read the last one
        if (threadIdx.x == 0)
            s_drawn = (int)atomicInc(out.long_tiles.taken + blockIdx.z, (uint32_t)items() + gridDim.x * (gridDim.y - out.long_rows) - 1);
        __syncthreads();
        return long_groups(out) + s_drawn;
    };
    for (int item = first ? long_group(out) : draw(); item < items(); item = draw()) {
        const TileId tile = tile_of_index(out.long_tiles.all[item / kMaxTileWaves]);
        const int part = item % kMaxTileWaves, n = a.offsets[tile.index + 1] - a.offsets[tile.index];
        if (n <= kShortList)
            long_tile_part<kSelectBatchShort, uint16_t, kHead, kPacked>(a, out, tile, part, s_dyn, nullptr);
        else
            long_tile_part<kSelectBatchShort, int, kLongHead, kPacked>(a, out, tile, part, s_dyn, nullptr);
    }
}

}  // namespace tg
