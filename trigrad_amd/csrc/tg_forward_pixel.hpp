// tg_forward_pixel.hpp -- the per-pixel-order forward kernel: selection and blending of one tile, the shared work of a long one.
// Its instances for launches whose workgroups all run at once are compiled in tg_forward_few.hip, those that read triangles' records in
// tg_forward_packed.hip, the others in tg_forward.hip.
#pragma once
#include "tg_forward.hpp"

namespace tg {

// render.cu:338-373 insert_sorted_topk on an LDS candidate list of capacity `cap`.
template <typename Pos>
__device__ __forceinline__ void topk_insert_at(const TopKOf<Pos> &tk, int i, real d, int j) {  // place i is free
    while (i > 0 && d < tk.d(i - 1)) {
        tk.d(i) = tk.d(i - 1);
        tk.j(i) = tk.j(i - 1);
        i--;
    }
    tk.d(i) = d;
    tk.j(i) = (Pos)j;
}
// last: the last candidate's depth.  A tile's list is sorted by depth, if not by the pixel's, so most candidates go behind the last
// one, and with its depth in a register that is a comparison and two writes, no read to wait for.
// Forward kernel, us, with the depth read from LDS for every candidate and so: 10^6 triangles 527, 487, 20 000 large ones without a
// limit on the layers 353, 309, 10^5 79, 72, 200 000 faint ones 289, 275, a mesh of 1.3 million 281, 273.
template <typename Pos>
__device__ __forceinline__ void topk_insert(const TopKOf<Pos> &tk, int cap, int &n, real &last, real d, int j) {
    const bool in_front = n > 0 && d < last;
    if (n < cap && !in_front) {
        tk.d(n) = d;
        tk.j(n) = (Pos)j;
        last = d;
        n++;
        return;
    }
    if (n == cap && d >= last) return;
    topk_insert_at(tk, (n < cap) ? n : cap - 1, d, j);
    if (n < cap) n++;
    else last = tk.d(cap - 1);
}

constexpr int kSelectBatch = 128;       // list entries staged per batch where positions take an int
constexpr int kSelectBatchShort = 64;   // ... and where they take 16 bits
// Places of a candidate list in LDS where positions take 16 bits; the rest is in registers (Candidates).  With 23 a workgroup of
// 256 threads takes 39.4 KB, four a CU, and fits the 128 registers of four waves per SIMD, where 32 were three: 10^6 triangles
// 601 -> 537 us, 10^5 92 -> 82, 20 000 large ones without a limit on the layers 431 -> 360, the mesh of 1.3 million 327 -> 297,
// 200 000 around the camera 117 -> 100, 33 000 in tiles of 8 x 8 (a wave to a workgroup) 88 -> 84.  With 22: 548, 83, 372.
// Lists with depth bounds keep all places in LDS and three kinds of 16-bit positions lose there: 200 000 faint triangles 288
// us, with 29 places and three workgroups a CU 301, with 21 and four 338: every pixel has 32 candidates.
constexpr int kShortHead = sizeof(real) == 4 ? 23 : kLayers;
// Waves a SIMD that the registers of the instances with 16-bit positions are held to, by their places in LDS: what the kernel is
// compiled with, and what the choice between them counts on (candidate_places).
constexpr int short_list_waves(int head) { return head < kLayers ? 4 : 3; }
constexpr int kLongHead = 17;  // the same LDS with int positions, in long_tile_part
static_assert((sizeof(real) + sizeof(int)) * kLongHead <= (sizeof(real) + sizeof(uint16_t)) * kShortHead, "the same LDS");

// The last places of a candidate list, in registers: place kPlace and those behind it.  (A structure of its own for every place:
// of an array the compiler makes scratch memory.)
template <int kPlace, int kPlaces>
struct ListTail {
    real d;
    int j;
    ListTail<kPlace + 1, kPlaces> rest;
    // bit k of places: depth x belongs in place k or further to the front; all: it is less than every one of the `used` first
    __device__ __forceinline__ void compare(real x, int used, bool &all, uint32_t &places) const {
        rest.compare(x, used, all, places);
        all = all && (kPlace >= used || x < d);
        places |= all && kPlace <= used ? 1u << kPlace : 0u;
    }
    __device__ __forceinline__ void insert(uint32_t places, int used, real x, int xj, real front_d, int front_j) {
        const bool shifted = kPlace > 0 && kPlace <= used && (places >> (kPlace > 0 ? kPlace - 1 : 0) & 1), here = places >> kPlace & 1;
        const real my_d = d;
        const int my_j = j;
        d = shifted ? front_d : here ? x : my_d;
        j = shifted ? front_j : here ? xj : my_j;
        rest.insert(places, used, x, xj, my_d, my_j);
    }
    __device__ __forceinline__ void read(int place, real &x, int &xj) const {
        x = place == kPlace ? d : x;
        xj = place == kPlace ? j : xj;
        rest.read(place, x, xj);
    }
};
template <int kPlaces>
struct ListTail<kPlaces, kPlaces> {
    __device__ __forceinline__ void compare(real, int, bool &, uint32_t &) const {}
    __device__ __forceinline__ void insert(uint32_t, int, real, int, real, int) {}
    __device__ __forceinline__ void read(int, real &, int &) const {}
};

// A pixel's candidates in the per-pixel-order pass: the nearest kHead in LDS, the others (kLayers - kHead) in registers, which
// few pixels have and which only they pay for.  Insertion is topk_insert's, place by place: from the end of the list to the
// front, as far as the new depth is less.
template <typename Pos, int kHead>
struct Candidates {
    TopKOf<Pos> head;
    ListTail<0, kLayers - kHead> tail;

    __device__ __forceinline__ void insert(int cap, int &n, real &last, real d, int j) {
        if (kHead == kLayers || n < kHead || cap <= kHead) {  // fewer than kHead: there is a place, whichever of the two ends it is
            topk_insert(head, min(cap, kHead), n, last, d, j);
            return;
        }
        if (n == cap && d >= last) return;
        const int used = n == cap ? cap - 1 - kHead : n - kHead;  // a full list loses its last
        bool all = true;
        uint32_t places = 0;
        tail.compare(d, used, all, places);
        const real last_d = head.d(kHead - 1);
        const int last_j = head.j(kHead - 1);
        const bool to_head = all && d < last_d;  // then the tail takes the head's last one, in its first place
        tail.insert(places, used, to_head ? last_d : d, to_head ? last_j : j, 0.0f, 0);
        if (to_head) topk_insert_at(head, kHead - 1, d, j);
        if (n < cap) n++;
        last = depth(n - 1);
    }
    __device__ __forceinline__ real depth(int i) const {
        if constexpr (kHead == kLayers) return head.d(i);
        real d = head.d(min(i, kHead - 1));
        int j = 0;
        tail.read(i - kHead, d, j);
        return d;
    }
    template <bool kBranch>  // the wave has a branch, as few lists are longer than kHead; it costs two registers
    __device__ __forceinline__ int position(int i) const {
        if (kHead == kLayers || (kBranch && __builtin_amdgcn_ballot_w64(i >= kHead) == 0)) return head.j(i);
        int j = head.j(min(i, kHead - 1));
        real d = 0.0f;
        tail.read(i - kHead, d, j);
        return j;
    }
};

// The per-pixel-order forward pass of one tile.  Pos: how a candidate's list position (from the tile's
// start) is kept.  With uint16_t the candidate lists of a 16x16 tile take 48 KB instead of 64 KB, which
// together with 64 staged entries lets a CU hold three workgroups instead of two.
template <int kStage, typename Pos, bool kInTurn, int kHead, bool kPacked>  // kStage: list entries staged per batch
__device__ __forceinline__ void pixel_order_tile(const RasterArgs &a, const ForwardOut &out, int tile_x, int tile_y, int tiles_x, int n_tiles,
                                                 unsigned char *s_dyn, uint8_t *s_touch, WaveRect *s_rects) {
    const int n_threads = kInTurn ? kTileThreads : blockDim.x;
    DepthRecord *s_rec = reinterpret_cast<DepthRecord *>(s_dyn);
    Candidates<Pos, kHead> tk;
    tk.head.depth = reinterpret_cast<real *>(s_dyn + sizeof(DepthRecord) * kStage);
    tk.head.pos = reinterpret_cast<Pos *>(tk.head.depth + kHead * n_threads);
    tk.head.n_threads = n_threads;

    const int tid = threadIdx.x;
    const int wave = tid / kWave;
    const int n_waves = blockDim.x / kWave;
    const int tile = tile_y * tiles_x + tile_x;
    const int start = a.offsets[tile], end = a.offsets[tile + 1];
    const PixelCoord p = pixel_of_thread(a, tile_x, tile_y);
    publish_wave_rect(a, p, s_rects);
    const bool tests_small = tests_small_entries(a, end - start, n_tiles);
    const int64_t order_step = order_stride(out.order, a);
    const int64_t order_at = order_first(out.order, p, start, blockIdx.z * blockDim.x + threadIdx.x);

    const int rows_kept = out.order.low ? order_rows(out.order, a, end - start) : 0;
    PixelState s;
    real last_depth = -__builtin_inff();  // render.cu:585-586
    int last_j = -1;  // list positions count from the tile's start
    bool active = p.valid && start < end;  // below, a list has a last entry
    for (bool again = false; start < end; again = true) {
        const bool want = active && s.alpha > a.thr && s.blended < a.max_layers;  // render.cu:588
        // The first time all pixels want what one does.  And what one selection takes is all there is where no more layers are asked for:
        // a pixel with fewer candidates than that is through with its list.
        if (again && (a.max_layers <= kLayers || !__syncthreads_or(want))) break;
        const int cap = want ? min(kLayers, a.max_layers - s.blended) : 0;
        int found = 0;
        real found_depth = 0.0f;  // of the last candidate
        // The records of coming batches are fetched into registers while this batch is worked on.  A wave that asks for an
        // entry's vertices has to have its vertex numbers, and for those its triangle number: three memory latencies in a
        // row, and whoever asks waits for the first two.  So the four waves of a tile take the batches in turn (kInTurn;
        // batches of 128 two waves each), and a wave's links are asked for half a turn apart; each has arrived when the next
        // one needs it.  A frame with a list of 8400 entries in one tile: 241 -> 154 us; lists of 268 everywhere: 680 -> 669.
        // Where depth bounds make the batches jump the turns start again (200 000 faint triangles, lists of 3700: 306 -> 292).
        constexpr int kTurns = kTileThreads / kStage;
        const int group = kStage == kWave ? wave : tid / kStage, mine = tid & (kStage - 1);  // in turn: whose batch, which of its entries
        const bool ahead = !kInTurn && !a.batch_bounds && (int)blockDim.x >= kStage;
        std::conditional_t<kPacked, PackedParts, std::conditional_t<kStage == kWave, PlacedParts, DepthParts>> next;
        auto start_turns = [&](int first) {  // the records of the kTurns batches from list entry `first` on
            const int j = min(first + tid, end - 1);
            next.fetch_triangle(a, j);
            next.fetch_matrix(a);
            next.fetch_triangle(a, min(j + kTileThreads, end - 1));
            next.fetch_vertices(a);
        };
        if constexpr (kInTurn) {
            start_turns(start);
        } else if (ahead && tid < min(kStage, end - start)) {
            next.fetch_triangle(a, start + tid);
            next.fetch_matrix(a);
            next.fetch_vertices(a);
        }
        int turn = 0;
        for (int batch = start; batch < end; batch += kStage, turn = (turn + 1) & (kTurns - 1)) {
            const int nb = min(kStage, end - batch);
            if (kStage != kWave && a.batch_bounds) {  // batches of 64 go without
                // a lane needs nothing from here on when its list is full and its worst candidate is nearer than
                // every fragment the rest of the tile's list can produce (a full list rejects depths >= its worst)
                const real rest = a.batch_bounds[batch_bound_index(start, tile, batch - start)];
                const bool settled = !want || (found == cap && found_depth <= rest);
                if (__syncthreads_and(settled)) {
                    // on to the batch that holds the first entry the bounds do not cover
                    const int resume = start + a.far_start[tile] / kStage * kStage;
                    if (resume > batch) {
                        if (kInTurn) {
                            start_turns(resume);
                            turn = kTurns - 1;
                        }
                        batch = resume - kStage;
                        continue;
                    }
                }
            }
            __syncthreads();
            if (kInTurn ? group == turn && mine < nb : ahead && tid < nb) {
                const int e = kInTurn ? mine : tid;
                const DepthRecord r = next.record();
                s_rec[e] = r;
                s_touch[e] = (uint8_t)(waves_touched(r.m, s_rects, n_waves, next.reach(r)) | small_entry(a, r.extent, tests_small));
            }
            if (!kInTurn && !ahead) {
                for (int e = tid; e < nb; e += blockDim.x) {
                    const Reach reach = gather_depth<kPacked>(a, batch + e, s_rec[e]);
                    s_touch[e] = (uint8_t)(waves_touched(s_rec[e].m, s_rects, n_waves, reach) | small_entry(a, s_rec[e].extent, tests_small));
                }
            }
            __syncthreads();
            if constexpr (kInTurn) {
                if (group == turn) {
                    // my next batch: its triangle numbers are here; ask for vertex numbers and matrices, and for the triangle
                    // numbers of the batch after it (past the list's end: its last entry again, which nobody looks at)
                    next.fetch_matrix(a);
                    next.fetch_triangle(a, min(batch + 2 * kTileThreads + mine, end - 1));
                } else if (group == (turn ^ (kTurns / 2))) {
                    next.fetch_vertices(a);
                }
            } else if (ahead && batch + kStage < end && tid < min(kStage, end - batch - kStage)) {
                next.fetch_triangle(a, batch + kStage + tid);
                next.fetch_matrix(a);
                next.fetch_vertices(a);
            }
            // inside tests into a per-lane mask, then every lane visits its own hits in
            // list order (the order insert_sorted_topk sees them in the reference)
            uint64_t m[kStage / kWave];
            batch_hit_mask<kStage / kWave>(s_rec, s_touch, s_rects, nb, wave, p.px, p.py, m);
            if (!want) {
#pragma unroll
                for (int wd = 0; wd < kStage / kWave; wd++) m[wd] = 0;
            }
            while (any_set<kStage / kWave>(m)) {
                const int e = pop_lowest<kStage / kWave>(m);
                const DepthRecord &r = s_rec[e];
                real b0, b1, b2;
                bary_apply(r.m, p.px, p.py, b0, b1, b2);
                const real pd = interp_w(b0, b1, b2, r.z[0], r.z[1], r.z[2], r.w[0], r.w[1], r.w[2]);  // render.cu:404
                const int j = batch + e - start;
                if (pd < last_depth) continue;
                if (pd == last_depth && j <= last_j) continue;
                tk.insert(cap, found, found_depth, pd, j);
            }
        }
        // Selection is over: the staging area and the depth lists are dead apart from
        // the depth of the last fragment each lane is going to blend.  The space takes
        // the blend records of the first list entries (rows an odd number of words
        // apart: lanes reading different entries use different banks); entries
        // beyond it are gathered from memory.
        const int todo = (want && found > 0) ? min(found, a.max_layers - s.blended) : 0;
        const real todo_depth = found_depth;  // todo is all of them: room is what cap was made for
        __syncthreads();
        real *rows = reinterpret_cast<real *>(s_dyn);
        const int n_rows = min(end - start, (int)((sizeof(DepthRecord) * kStage + sizeof(real) * kHead * n_threads) /
                                                   (sizeof(real) * kBlendWords)));
        for (int e = tid; e < n_rows; e += blockDim.x) {
            BlendRecord r;
            gather_blend<kPacked>(a, start + e, r);
            const real *w = reinterpret_cast<const real *>(&r);
#pragma unroll
            for (int k = 0; k < kBlendWords; k++) rows[e * kBlendWords + k] = w[k];
        }
        __syncthreads();
        if (want) {
            if (found == 0) {
                active = false;  // render.cu:594
            } else {
                // kTogether records are fetched together: the chains of dependent loads (list -> indices -> vertices) of those
                // that come from memory overlap.  They are the kernel's peak of registers (two together where three would
                // do: lists of hundreds 220 -> 226)
                constexpr int kTogether = kHead < kLayers ? 1 : kInTurn ? 4 : 3;
                // one at a time, the next one's position is asked for while this one is blended, where there is a register left for it
                constexpr bool kAhead = kTogether == 1 && kInTurn;
                int ahead = kAhead ? tk.template position<kInTurn>(0) : 0;
                for (int i0 = 0; i0 < todo; i0 += kTogether) {
                    BlendRecord r[kTogether];
                    int rel[kTogether];
#pragma unroll
                    for (int u = 0; u < kTogether; u++) {
                        rel[u] = kAhead ? ahead : tk.template position<kInTurn>(kTogether == 1 ? i0 : min(i0 + u, todo - 1));
                        if (kAhead) ahead = tk.template position<kInTurn>(min(i0 + 1, kLayers - 1));
                        if (rel[u] < n_rows) {
                            const real *row = rows + __umul24((uint32_t)rel[u], kBlendWords);
                            real *w = reinterpret_cast<real *>(&r[u]);
#pragma unroll
                            for (int k = 0; k < kBlendWords; k++) w[k] = row[k];
                        } else {
                            gather_blend<kPacked>(a, start + rel[u], r[u]);
                        }
                    }
#pragma unroll
                    for (int u = 0; u < kTogether; u++) {
                        if (i0 + u >= todo) break;
                        real b0, b1, b2;
                        bary_apply(r[u].m, p.px, p.py, b0, b1, b2);
                        if (s.blended < rows_kept) {
                            const int64_t at = order_at + (int64_t)s.blended * order_step;
                            out.order.low[at] = (uint16_t)rel[u];
                            if (sizeof(Pos) > sizeof(uint16_t) && end - start > kShortList)
                                out.order.low[out.order.high + at] = (uint16_t)(rel[u] >> 16);
                        }
                        blend_fragment(s, r[u], b0, b1, b2);
                    }
                }
                last_depth = todo_depth;
                last_j = tk.template position<kInTurn>(todo - 1);
                // fewer candidates than asked for: the list is exhausted, the next
                // selection would return nothing (render.cu:594)
                if (found < cap) active = false;
            }
        }
    }
    if (p.valid) write_pixel(out, p, s, last_j + 1, last_depth);
}

// Visits the nearest `cap` candidates of a lane's pixel in the four waves' sorted lists, nearest first, by depth and list
// position: visit(i, depth, position).  short_list: a list was through before that which has dropped candidates.
// -> how many were visited.
template <typename Shared, typename Pos, typename Visit>
__device__ __forceinline__ int merge_lists(const Shared *shared, const TopKOf<Pos> &tk, int lane, int cap, Visit visit, bool &short_list) {
    const auto depth_at = [&](int w, int i) { return tk.depth[i * tk.n_threads + w * kWave + lane]; };
    const auto pos_at = [&](int w, int i) { return (int)tk.pos[i * tk.n_threads + w * kWave + lane]; };
    uint32_t left = 0, at = 0;  // of every list: candidates not visited yet, and the next one's place; a byte each
    int pos[kMaxTileWaves];
    real depth[kMaxTileWaves];
    uint32_t dropped = 0;
#pragma unroll
    for (int w = 0; w < kMaxTileWaves; w++) {
        const int count = shared->found[w * kWave + lane];
        left |= (uint32_t)count << (8 * w);
        dropped |= (uint32_t)shared->dropped[w * kWave + lane] << w;
        depth[w] = count ? depth_at(w, 0) : 0.0f;
        pos[w] = count ? pos_at(w, 0) : 0;
    }
    for (int i = 0; i < cap; i++) {
        int best = -1, j = 0;
        real d = 0.0f;
#pragma unroll
        for (int w = 0; w < kMaxTileWaves; w++) {
            if ((left >> (8 * w) & 0xff) == 0) {
                short_list = short_list || (dropped >> w & 1);
            } else if (best < 0 || depth[w] < d || (depth[w] == d && pos[w] < j)) {
                best = w;
                d = depth[w];
                j = pos[w];
            }
        }
        if (best < 0) return i;
        visit(i, d, j);
        left -= 1u << (8 * best);
        at += 1u << (8 * best);
#pragma unroll
        for (int w = 0; w < kMaxTileWaves; w++)
            if (w == best && (left >> (8 * w) & 0xff)) {
                depth[w] = depth_at(w, at >> (8 * w) & 0xff);
                pos[w] = pos_at(w, at >> (8 * w) & 0xff);
            }
    }
    return cap;
}

// A wave's share (64 pixels; the part-th of its workgroup's) of a tile with a long list, by the four waves of a workgroup: each
// takes every fourth entry and keeps candidate lists of its own, without a barrier, and the first wave merges the
// four sorted lists of a pixel, by depth and list position, while it blends.  A list was one workgroup's serial chain before,
// 7 us for every 64 entries with most of the CU empty; it is a quarter as long now, and a tile's four squares run beside
// each other.  What a wave tests it holds in registers, lane = entry, so only the entries that are hit go through LDS, kStage / 4
// at a time: the candidate lists leave no more (64 at a time, with fewer candidates kept, is no faster).
// 1.3 million triangles of a mesh, 1920 x 1080 (longest list 5200, 221 of at least 1024): 604 -> 332 us; 200 000 around the
// camera (one list of 8400): 152 -> 117; 81 tiles with lists of some 2600, where depth bounds end the looking early: 105 -> 91.
// s_quarter: a depth for every thread, with depth bounds; else null.
template <int kStage, typename Pos, int kHead, bool kPacked>
__device__ __forceinline__ void long_tile_part(const RasterArgs &a, const ForwardOut &out, const TileId &tile, int part, unsigned char *s_dyn,
                                               volatile real *s_quarter) {
    constexpr int kStaged = kStage / kMaxTileWaves;  // records of a wave in LDS at a time
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));  // what depends on it is made here, not kept in registers by the loop around the call
    const int lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int start = a.offsets[tile.index], end = a.offsets[tile.index + 1], n = end - start;
    DepthRecord *s_rec = reinterpret_cast<DepthRecord *>(s_dyn) + wave * kStaged;
    TopKOf<Pos> tk;
    tk.depth = reinterpret_cast<real *>(s_dyn + sizeof(DepthRecord) * kStage);
    tk.pos = reinterpret_cast<Pos *>(tk.depth + kHead * kTileThreads);
    static_assert(kLayers <= kMaxTileWaves * kHead, "one wave's lists have room in the place of four");
    // between two selections the place of the staged records holds what the waves tell each other
    struct Shared { int found[kTileThreads], cap[kWave], last_j[kWave], again[kMaxTileWaves]; real last_depth[kWave]; uint8_t dropped[kTileThreads]; };
    static_assert(sizeof(Shared) <= sizeof(DepthRecord) * kStage, "the waves' exchange fits the staging area");
    Shared *shared = reinterpret_cast<Shared *>(s_dyn);

    const int slot = (blockIdx.z * kMaxTileWaves + part) * kWave + lane;
    const PixelCoord p = pixel_of_slot(a, tile.x, tile.y, slot);
    const WaveRect rect = wave_rect(a, p);
    const bool squares = ((a.tw | a.th) & 7) == 0;

    PixelState s;  // of the first wave
    real last_depth = -__builtin_inff();
    int last_j = -1;
    bool active = p.valid && n > 0;
    while (true) {
        const int wanted = active && s.alpha > a.thr && s.blended < a.max_layers ? min(kLayers, a.max_layers - s.blended) : 0;
        __syncthreads();
        if (wave == 0) {
            shared->cap[lane] = wanted;
            shared->last_depth[lane] = last_depth;
            shared->last_j[lane] = last_j;
        }
        if (s_quarter) s_quarter[tid] = __builtin_inff();
        __syncthreads();
        const int cap = shared->cap[lane];
        last_depth = shared->last_depth[lane];
        last_j = shared->last_j[lane];
        if (__builtin_amdgcn_ballot_w64(cap > 0) == 0) break;  // the same for all waves
        __syncthreads();
        // The waves take the list's entries in turn, each with candidate lists of its own, of kHead places.  (Not blocks of 64: the
        // list is sorted by depth, so where triangles cover the square a pixel's nearest candidates are in one block, one wave's,
        // which drops some: 30 tiles of 3000 large faint triangles among 60 000 small ones 750 us, by entries 294, one workgroup a
        // tile 562.)  Where that does not do the first wave makes the selection alone, with room for all the layers: if a wave dropped a candidate
        // that may be among the nearest (the merge comes to the end of its list); and if a depth is NaN, which ends a candidate
        // list wherever it comes (topk_insert), so that what stays depends on what came before it.
        int found = 0, todo = 0;
        for (int waves = kMaxTileWaves; ; waves = 1) {
            tk.n_threads = waves == 1 ? kWave : kTileThreads;
            const int room = min(cap, waves == 1 ? kLayers : kHead);
            found = 0;
            bool met_nan = false, dropped = false;
            real found_depth = 0.0f;
            if (wave < waves) {
                // a group of the list is 64 entries for each wave
                const int group = waves * kWave, mine = lane * waves + wave;
                const auto entry = [&](int first) { return min(start + first + mine, end - 1); };
                std::conditional_t<kPacked, PackedParts, DepthParts> next;
                const auto fetch_from = [&](int first) {
                    next.fetch_triangle(a, entry(first));
                    next.fetch_matrix(a);
                    next.fetch_triangle(a, entry(first + group));
                    next.fetch_vertices(a);
                };
                fetch_from(0);
                for (int first = 0; first < n; first += group) {
                    if (kStage != kWave && a.batch_bounds) {
                        // as in pixel_order_tile: there are enough candidates nearer than all the rest of the list.  Each wave
                        // knows that of a quarter of them in every wave's lists; at a depth of its own the rest might come
                        // before another wave's candidate.
                        const real rest = a.batch_bounds[batch_bound_index(start, tile.index, first)];
                        const int resume = a.far_start[tile.index] / group * group;
                        bool settled = cap == 0;
                        if (!settled && waves == 1) settled = found == room && found_depth <= rest;
                        if (!settled && waves > 1) {
                            settled = true;
#pragma unroll
                            for (int w = 0; w < kMaxTileWaves; w++) settled = settled && s_quarter[w * kWave + lane] < rest;
                        }
                        if (resume > first && !__builtin_amdgcn_ballot_w64(!settled)) {
                            first = resume;
                            if (first >= n) break;
                            fetch_from(first);
                        }
                    }
                    const DepthRecord r = next.record();
                    next.fetch_matrix(a);
                    next.fetch_triangle(a, entry(first + 2 * group));
                    uint64_t hit;
                    uint64_t m = wave_hits(r.m, first + mine < n, squares, rect, p.px, p.py, hit);
                    if (cap == 0) m = 0;
                    next.fetch_vertices(a);
                    while (hit) {  // wave-uniform: the hit entries' records through LDS, kStaged at a time
                        const uint32_t rank = lanes_below_mask(hit);
                        const bool staged = ((hit >> lane) & 1) && rank < (uint32_t)kStaged;
                        const uint64_t there = __builtin_amdgcn_ballot_w64(staged);
                        if (staged) s_rec[rank] = r;
                        wave_lds_sync();
                        uint64_t todo = m & there;
                        while (__builtin_amdgcn_ballot_w64(todo != 0)) {
                            if (todo == 0) continue;
                            const int e = __builtin_ctzll(todo);
                            todo &= todo - 1;
                            const DepthRecord &d = s_rec[__builtin_popcountll(there & ((1ull << e) - 1))];
                            real b0, b1, b2;
                            bary_apply(d.m, p.px, p.py, b0, b1, b2);
                            const real pd = interp_w(b0, b1, b2, d.z[0], d.z[1], d.z[2], d.w[0], d.w[1], d.w[2]);  // render.cu:404
                            const int j = first + e * waves + wave;
                            met_nan = met_nan || pd != pd;
                            if (pd < last_depth || (pd == last_depth && j <= last_j)) continue;
                            dropped = dropped || (found == room && room < cap);
                            topk_insert(tk, room, found, found_depth, pd, j);
                        }
                        hit &= ~there;
                        wave_lds_sync();
                    }
                    const int quarter = (cap + kMaxTileWaves - 1) / kMaxTileWaves;
                    if (s_quarter && waves > 1 && cap > 0 && found >= quarter) s_quarter[tid] = tk.d(quarter - 1);
                }
            }
            __syncthreads();
            shared->found[tid] = found;
            shared->dropped[tid] = dropped;
            const uint64_t nan_lanes = __builtin_amdgcn_ballot_w64(met_nan);
            if (lane == 0) shared->again[wave] = waves > 1 && nan_lanes != 0;
            __syncthreads();
            if (wave == 0 && waves > 1) {
                bool short_list = false;
                merge_lists(shared, tk, lane, cap, [&](int, real, int) {}, short_list);
                const uint64_t short_lanes = __builtin_amdgcn_ballot_w64(short_list);
                if (lane == 0 && short_lanes) shared->again[0] = 1;
            }
            __syncthreads();
            const int again = shared->again[0] | shared->again[1] | shared->again[2] | shared->again[3];
            __syncthreads();
            if (!again) break;
        }
        if (wave == 0 && cap > 0) {
            const int64_t order_step = order_stride(out.order, a);
            const int64_t order_at = order_first(out.order, p, start, slot);
            const int rows_kept = out.order.low ? order_rows(out.order, a, n) : 0;
            bool short_list = false;
            todo = merge_lists(shared, tk, lane, cap, [&](int, real d, int j) {
                last_depth = d;
                last_j = j;
                BlendRecord r;
                gather_blend<kPacked>(a, start + j, r);
                if (s.blended < rows_kept) {
                    const int64_t word = order_at + (int64_t)s.blended * order_step;
                    out.order.low[word] = (uint16_t)j;
                    if (sizeof(Pos) > sizeof(uint16_t) && n > kShortList) out.order.low[out.order.high + word] = (uint16_t)(j >> 16);
                }
                real b0, b1, b2;
                bary_apply(r.m, p.px, p.py, b0, b1, b2);
                blend_fragment(s, r, b0, b1, b2);
            }, short_list);
            if (todo < cap) active = false;  // the list is exhausted (render.cu:594)
        }
    }
    if (wave == 0 && p.valid) write_pixel(out, p, s, last_j + 1, last_depth);
}

// One workgroup per tile.  With 16-bit positions the tiles whose lists are too long for them are shared out as long tiles, with
// int positions, or left to forward_pixel_order_long_lists_kernel.
// kInTurn: the workgroup has four waves.
// Workgroups a CU: what their LDS allows.  No bound in double precision: held to two workgroups every instance spills (10^5
// triangles, 1024 x 1024: 229 us instead of 223, tiles of 8 x 8 190 instead of 168).
template <int kStage, typename Pos, bool kInTurn, int kHead, bool kPacked>
__global__ __launch_bounds__(kTileThreads, sizeof(real) != 4 ? 1 : kStage != kSelectBatchShort ? 2 : short_list_waves(kHead))
void forward_pixel_order_kernel(RasterArgs a, ForwardOut out) {
    extern __shared__ __align__(16) unsigned char s_dyn[];
    __shared__ uint8_t s_touch[kStage];
    __shared__ WaveRect s_rects[kMaxTileWaves];
    if (lists_invalid(out)) {  // the same for the whole launch
        mark_tile_invalid(a, out);
        return;
    }
    const bool first = (int)blockIdx.y < out.long_rows;
    if constexpr (kInTurn && kSharesLongTiles) {
        if (first) {
            __shared__ real s_quarter[kStage != kWave ? kTileThreads : 1];  // with depth bounds; batches of 64 go without
            const int n_items = kMaxTileWaves * out.long_tiles.words[0];
            for (int item = long_group(out); item < n_items; item += long_groups(out)) {
                const TileId tile = tile_of_index(out.long_tiles.all[item / kMaxTileWaves]);
                const int part = item % kMaxTileWaves, n = a.offsets[tile.index + 1] - a.offsets[tile.index];
                if (sizeof(Pos) == sizeof(int) || n <= kShortList)
                    long_tile_part<kStage, Pos, kHead, kPacked>(a, out, tile, part, s_dyn, kStage != kWave ? s_quarter : nullptr);
                else
                    long_tile_part<kStage, int, kLongHead, kPacked>(a, out, tile, part, s_dyn, nullptr);
            }
            return;
        }
    } else {
        if (first && long_group(out) >= tiles_started_first(out)) return;
    }
    const TileId tile = first ? tile_of_index(out.long_tiles.words[1 + long_group(out)]) : tile_of_workgroup<kTileBandForward, kChunkForward>(out.long_rows);
    const int n_entries = a.offsets[tile.index + 1] - a.offsets[tile.index];
    if (sizeof(Pos) < sizeof(int) && n_entries > kShortList) return;
    if (kInTurn ? is_long_tile(out, n_entries) : !first && is_started_first(out, tile.index, n_entries)) return;
    pixel_order_tile<kStage, Pos, kInTurn, kHead, kPacked>(a, out, tile.x, tile.y, gridDim.x, gridDim.x * (gridDim.y - out.long_rows), s_dyn, s_touch, s_rects);
}

constexpr int kLongListGroups = 256;    // workgroups that look for the tiles with longer lists

// The tiles whose lists are longer than kShortList, with int positions, where forward_pixel_order_kernel does not share them out as long
// tiles (their launch is saved there, 4.7 us whether there are any or not): few or none, so a small grid looks through the
// tiles' list lengths (a workgroup through its share of the tiles, one tile per thread at a time) and takes those.
template <bool kPacked>
__global__ __launch_bounds__(kTileThreads) void forward_pixel_order_long_lists_kernel(RasterArgs a, ForwardOut out, int tiles_x,
                                                                                      int tiles_y) {
    extern __shared__ __align__(16) unsigned char s_dyn[];
    __shared__ uint8_t s_touch[kSelectBatch];
    __shared__ WaveRect s_rects[kMaxTileWaves];
    __shared__ uint64_t s_votes[kMaxTileWaves];
    if (out.list_status && *out.list_status != TG_STATUS_OK) return;  // the launch before this one has marked every pixel
    const int tiles = tiles_x * tiles_y;
    const int share = (tiles + (int)gridDim.x - 1) / (int)gridDim.x;
    const int first = blockIdx.x * share, past = min(first + share, tiles);
    const int n_waves = blockDim.x / kWave;
    for (int base = first; base < past; base += blockDim.x) {
        const int mine = base + (int)threadIdx.x;
        const int length = mine < past ? a.offsets[mine + 1] - a.offsets[mine] : 0;
        const bool is_long = length > kShortList && !(out.long_rows && blockDim.x == kTileThreads && length >= out.long_tiles.limit);
        const uint64_t vote = __builtin_amdgcn_ballot_w64(is_long);
        __syncthreads();  // the round before is done with the votes
        if ((threadIdx.x & (kWave - 1)) == 0) s_votes[threadIdx.x / kWave] = vote;
        __syncthreads();
        for (int w = 0; w < n_waves; w++) {
            uint64_t todo = s_votes[w];
            while (todo) {  // the same for the whole workgroup
                const int tile = base + w * kWave + __builtin_ctzll(todo);
                todo &= todo - 1;
                __syncthreads();  // the tile before is done with the LDS
                pixel_order_tile<kSelectBatch, int, false, kLayers, kPacked>(a, out, tile % tiles_x, tile / tiles_x, tiles_x, tiles, s_dyn, s_touch, s_rects);
            }
        }
    }
}

}  // namespace tg
