// tg_raster.hpp -- pieces shared by the forward and backward tile kernels.
//
// Launch shape: grid (tiles_x, tiles_y, parts); a workgroup of at most 256 threads
// owns pixels [part*blockDim, (part+1)*blockDim) of its tile, so tiles of more are split into several
// workgroups that walk the same list.
// Forward, and backward where no blend order was saved: a 16x16 tile is exactly one workgroup of four waves, part = z.
// The tile's sorted list is consumed in batches: up to kBatch threads each gather one list entry (triangle id ->
// vertex ids -> vertex data, bary matrix, attributes) into an LDS record, then
// every pixel thread walks the records; all lanes read the same record at the
// same time, which LDS serves as a broadcast.
// The two other backward kernels: a wave works by itself, a workgroup is one or four of them (part_of_workgroup), and nothing is
// staged; a fragment's record is gathered where the fragment is evaluated.
#pragma once
#include "tg_common.hpp"

namespace tg {

constexpr int kBatch = 128;         // list entries staged per batch
constexpr int kBoundSpan = 256;     // list entries per depth bound (tg_list_bounds)
constexpr int kLayers = 32;         // per-pixel selection batch (render.cu:570, :655)
constexpr int kMaxTilePixels = 1024;  // tile_w * tile_h limit of the API (wrapper.py:143)
constexpr int kTileThreads = 256;     // workgroup size limit
constexpr bool kPacks = sizeof(real) == 4;  // records are what a frame in one call has, a call of the float build
constexpr int kShortList = 0xffff;    // longest tile list whose positions fit 16 bits

struct RasterArgs {
    const real4 *vertices;
    const int32_t *indices;
    const real *colors;
    const real *opacities;
    const int32_t *sorted_ids;
    const int32_t *offsets;
    const real *bary;
    const real *batch_bounds;  // per tile and kBoundSpan entries: lower bound of the pixel depths from there on; may be null
    const int32_t *far_start;  // per tile: first list position whose entries the bounds do not cover (with batch_bounds)
    int W, H, tw, th;
    real thr;
    int max_layers;
    const real4 *records = nullptr;  // one TriangleRecord per triangle, for the instances that are packed
};

struct PixelCoord {
    int ix, iy, index;
    bool valid;
    real px, py;
};

// x / d and x % d for a d that is the same for the wave and mostly a power of two: a division is twenty operations.
__device__ __forceinline__ void divide(int x, int d, int &quotient, int &rest) {  // x >= 0, d > 0
    if ((d & (d - 1)) == 0) {
        quotient = x >> __builtin_ctz(d);
        rest = x & (d - 1);
    } else {
        quotient = x / d;
        rest = x - quotient * d;
    }
}

// The pixel in slot t of a tile.
__device__ __forceinline__ PixelCoord pixel_of_slot(const RasterArgs &a, int tile_x, int tile_y, int t) {
    PixelCoord p;
    int lx, ly;
    if (((a.tw | a.th) & 7) == 0) {
        // a wave takes a square of 8 x 8 pixels: fewer list entries touch a square than a strip of the
        // same area, so the waves cull more and share an entry among more lanes
        int squares_x = a.tw >> 3;
        asm volatile("" : "+s"(squares_x));  // the division's constants are made here, not kept in registers by a loop around the call
        const int square = t >> 6, l = t & 63;
        int row, column;
        divide(square, squares_x, row, column);
        lx = column * 8 + (l & 7);
        ly = row * 8 + (l >> 3);
    } else {
        int columns = a.tw;
        asm volatile("" : "+s"(columns));
        lx = t % columns;
        ly = t / columns;
    }
    p.ix = tile_x * a.tw + lx;
    p.iy = tile_y * a.th + ly;
    p.valid = (t < a.tw * a.th) && p.ix < a.W && p.iy < a.H;  // render.cu:554
    p.index = p.iy * a.W + p.ix;
    p.px = pixel_ndc(p.ix, a.W);
    p.py = pixel_ndc(p.iy, a.H);
    return p;
}

__device__ __forceinline__ PixelCoord pixel_of_thread(const RasterArgs &a, int tile_x, int tile_y) {
    return pixel_of_slot(a, tile_x, tile_y, blockIdx.z * blockDim.x + threadIdx.x);
}

// The tile a workgroup of a (tiles_x, tiles_y, parts) launch takes.  Workgroups go to the eight XCDs of the device in
// turn in the order of their linear index, and every XCD has an L2 of its own; neighbouring tiles share list
// entries (a triangle that covers two tiles is in both lists), vertices and matrices.  So the workgroups
// that reach one XCD take consecutive tiles of an order that keeps neighbours together: bands of kTileBand
// tile rows, column by column inside a band.  The workgroups that run on an XCD at one time cover a compact block of the
// image.  Backward, XCD k gets the k-th eighth of that order.  Forward, the order is dealt out in chunks of kChunkForward tiles:
// where a mesh covers part of the image an eighth can be empty and another one full (1.3 million triangles of a torus,
// 1920 x 1080: two XCDs had 45 % of the list entries, the last one none; 800 -> 680 us of kernel time), and where every tile
// has the same work nothing is lost (10^6 triangles: 677 -> 668; chunks of 16 to 128 within 1 %).
// The backward kernel with the saved order takes two sixteenths, the k-th from either end: what lies in the middle, or on one side, is
// shared by all, and neighbours stay together nearly as well.  Frames, us, in eighths and so: mesh of 1.3 million triangles 734, 721,
// 20 000 large triangles on 512 x 512 1059, 1005, 10^6 triangles 1924, 1912 (in chunks of 16 tiles 716, 1008, 1936).
// Gradients that tiles on two XCDs share cost more than those that stay on one.  Deep enough that does not show; with few layers
// or short lists most of them are a few large triangles', which cover many tiles: 10^6 triangles with a heavy tail and 2, 8 layers
// 147, 577 us in eighths and 187, 604 in chunks; 900 and 7500 triangles with a heavy tail on 1920 x 1080, lists of 12, 682, 394 in
// eighths, 870, 485 in sixteenths.  So below kManyLayers layers or kDeepLists entries a tile (from there on 1.002 of the eighths' time
// on average over frames of all kinds, 1.08 at worst) it takes eighths, like the kernel in tile order, where vertices share lines
// in dense gradient arrays as well (618 -> 700 with chunks of 16).
#ifndef TG_XCD_TILES
#define TG_XCD_TILES 1
#endif
#ifndef TG_TILE_BAND_FORWARD
#define TG_TILE_BAND_FORWARD 8
#endif
#ifndef TG_TILE_BAND_BACKWARD
#define TG_TILE_BAND_BACKWARD 1
#endif
#ifndef TG_XCD_CHUNK_FORWARD
#define TG_XCD_CHUNK_FORWARD 32
#endif
constexpr int kXcds = 8;
constexpr int kTileBandForward = TG_TILE_BAND_FORWARD, kTileBandBackward = TG_TILE_BAND_BACKWARD;
constexpr int kEighths = 0, kSixteenths = -1;  // in the place of a number of tiles: one eighth of them an XCD, two sixteenths
constexpr int kChunkForward = TG_XCD_CHUNK_FORWARD;
constexpr int kManyLayers = 16, kDeepLists = 96;
struct TileId { int x, y, index; };
template <int kTileBand, int kChunk>
__device__ __forceinline__ TileId tile_in_turn(int linear, int tiles_x, int tiles_y) {
    const int n = tiles_x * tiles_y;
    TileId t;
#if TG_XCD_TILES
    const int xcd = linear % kXcds, turn = linear / kXcds;
    int place, first = 0, left = turn;  // first: what the rounds of whole chunks take; left: turns after them
    if (kChunk > 0) {
        const int round = turn / kChunk;
        first = round * kXcds * kChunk;
        left -= round * kChunk;
    }
    if (kChunk == kSixteenths) {
        const int part = n / (2 * kXcds);  // the last tiles, fewer than 16, go as they come
        place = turn < part ? xcd * part + turn : turn < 2 * part ? (2 * kXcds - 2 - xcd) * part + turn : linear;
    } else if (kChunk > 0 && first + kXcds * kChunk <= n) {
        place = first + xcd * kChunk + left;
    } else {
        const int per = (n - first) / kXcds, rest = (n - first) % kXcds;
        place = first + (xcd < rest ? xcd * (per + 1) + left : rest * (per + 1) + (xcd - rest) * per + left);
    }
    const int band = place / (kTileBand * tiles_x), within = place - band * (kTileBand * tiles_x);
    const int rows = min(kTileBand, tiles_y - band * kTileBand);
    int row;
    divide(within, rows, t.x, row);
    t.y = band * kTileBand + row;
#else
    t.x = linear % tiles_x;
    t.y = linear / tiles_x;
#endif
    t.index = t.y * tiles_x + t.x;
    return t;
}
template <int kTileBand, int kChunk>
__device__ __forceinline__ TileId tile_of_workgroup(int skipped_rows = 0) {  // rows of workgroups in front that are not for tiles
    return tile_in_turn<kTileBand, kChunk>((int)((blockIdx.y - skipped_rows) * gridDim.x + blockIdx.x), (int)gridDim.x, (int)gridDim.y - skipped_rows);
}
// A launch of gridDim.z workgroups a tile, of which those of one tile follow each other on its XCD: the place of the calling workgroup's
// tile in the order above, and which of the tile's workgroups it is.
struct TilePart { int linear, part; };
__device__ __forceinline__ TilePart part_of_workgroup() {
    const int tiles = (int)(gridDim.x * gridDim.y), parts = (int)gridDim.z;
    const int group = (int)((blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x);
    const int whole = tiles / kXcds * kXcds;  // the last tiles, fewer than eight, go as they come
    if (group >= whole * parts) {
        const int rest = group - whole * parts;
        return {whole + rest % (tiles - whole), rest / (tiles - whole)};
    }
    const int turn = group / kXcds;
    return {turn / parts * kXcds + group % kXcds, turn % parts};
}
__device__ __forceinline__ PixelCoord pixel_of_thread(const RasterArgs &a, const TileId &t) { return pixel_of_thread(a, t.x, t.y); }

// Everything process_forward (render.cu:417-453) reads for one list entry.
struct alignas(16) BlendRecord {
    real m[9];
    real w[3];
    real iw[3];   // 1/w per vertex (render.cu:444)
    real op[3];
    real col[9];  // vertex a rgb, vertex b rgb, vertex c rgb
    real extent;  // of the vertices in y (see small_entry)
};
static_assert(sizeof(BlendRecord) == 28 * sizeof(real), "BlendRecord layout");
constexpr int kBlendWords = 27;  // scalars of a BlendRecord without its padding; odd

// What select_next_k_in_tile (render.cu:375-415) reads for one list entry.
struct alignas(16) DepthRecord {
    real m[9];
    real z[3];
    real w[3];
    real extent;
};
static_assert(sizeof(DepthRecord) == 16 * sizeof(real), "DepthRecord layout");

struct TriIds { int tri, ia, ib, ic; };

__device__ __forceinline__ TriIds load_ids(const RasterArgs &a, int j) {
    TriIds t;
    t.tri = a.sorted_ids[j];
    t.ia = a.indices[3 * (int64_t)t.tri];
    t.ib = a.indices[3 * (int64_t)t.tri + 1];
    t.ic = a.indices[3 * (int64_t)t.tri + 2];
    return t;
}

// The attributes of a record's vertices.
__device__ __forceinline__ void gather_attributes(const RasterArgs &a, int ia, int ib, int ic, BlendRecord &r) {
    r.op[0] = a.opacities[ia]; r.op[1] = a.opacities[ib]; r.op[2] = a.opacities[ic];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        r.col[k] = a.colors[3 * (int64_t)ia + k];
        r.col[3 + k] = a.colors[3 * (int64_t)ib + k];
        r.col[6 + k] = a.colors[3 * (int64_t)ic + k];
    }
}

__device__ __forceinline__ float min_number(float a, float b, float c) { return __builtin_fminf(__builtin_fminf(a, b), c); }
__device__ __forceinline__ double min_number(double a, double b, double c) { return __builtin_fmin(__builtin_fmin(a, b), c); }
__device__ __forceinline__ float max_number(float a, float b, float c) { return __builtin_fmaxf(__builtin_fmaxf(a, b), c); }
__device__ __forceinline__ double max_number(double a, double b, double c) { return __builtin_fmax(__builtin_fmax(a, b), c); }

// Bounds of the pixel centres that an entry's inside tests can let in, besides those of its edges (may_touch).
//
// The tests are of the matrix m (rows b_k = m_k0 x + m_k1 y + m_k2), which is the inverse of the vertices' up to rounding, so
// what it really says of x is looked at.  For a pixel inside, every b_k >= 0 as computed, so in exact arithmetic
// b_k >= -3u S_k, where S_k = |m_k0| + |m_k1| + |m_k2|, u is half an epsilon and |x|, |y| <= 1.  Times x_k - x_min >= 0 and summed:
//     x - x_min + r(x, y) + (x_0 - x_min) s(x, y) >= -3u w S,   S = sum of S_k, w = x_max - x_min,
//     s = sum of b_k - 1,  r = sum of (x_k - x_0) b_k - (x - x_0),
// both zero if m were the inverse.  With the absolute sums of their coefficients for |r| and |s|, rounded by less than
// 9u (w S + |x_0| + 1) together, x >= x_min - (|r| + w |s|) - 12u (w S + |x_0| + 1); a hundredth more and 32u (w S + 1) are more than
// that and the rounding of the bound itself (|x_0| <= w + 1, and S + |s| >= 1, unless all vertices are on one side of the screen, and
// then a bound near the screen is a margin near |x_0|, with the hundredth).  The same for x_max and for y.  A margin is a tenth of a
// pixel or less for triangles of some pixels; a matrix that is no inverse, overflows or is NaN makes bounds that leave nothing out.
struct Reach { real x_lo, x_hi, y_lo, y_hi; };
__device__ __forceinline__ Reach reaches_everywhere() {
    constexpr real kFar = std::numeric_limits<real>::infinity();
    return Reach{-kFar, kFar, -kFar, kFar};
}
__device__ __forceinline__ float fused(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fused(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float size_of(float a) { return __builtin_fabsf(a); }
__device__ __forceinline__ double size_of(double a) { return __builtin_fabs(a); }
__device__ __forceinline__ real sum3(real a, real b, real c) { return size_of(a) + size_of(b) + size_of(c); }
__device__ __forceinline__ void reach_along(const real m[9], real a, real b, real c, bool along_y, real strayed, real size, real &lo, real &hi) {
    const real db = b - a, dc = c - a;
    const real r0 = fused(db, m[3], fused(dc, m[6], along_y ? (real)0.0f : (real)-1.0f));
    const real r1 = fused(db, m[4], fused(dc, m[7], along_y ? (real)-1.0f : (real)0.0f));
    const real r2 = fused(db, m[5], fused(dc, m[8], a));
    const real least = min_number(a, b, c), most = max_number(a, b, c), w = most - least;
    const real margin = fused(sum3(r0, r1, r2), (real)1.01, fused(w, fused(strayed, (real)1.01, size), (real)(16 * std::numeric_limits<real>::epsilon())));
    lo = least - margin;
    hi = most + margin;
}
__device__ __forceinline__ Reach triangle_reach(const real m[9], real ax, real ay, real bx, real by, real cx, real cy) {
    const real strayed = sum3(m[0] + m[3] + m[6], m[1] + m[4] + m[7], m[2] + m[5] + m[8] - 1.0f);
    const real size = (sum3(m[0], m[1], m[2]) + sum3(m[3], m[4], m[5]) + sum3(m[6], m[7], m[8])) * (16 * std::numeric_limits<real>::epsilon());
    Reach r;
    reach_along(m, ax, bx, cx, false, strayed, size, r.x_lo, r.x_hi);
    reach_along(m, ay, by, cy, true, strayed, size, r.y_lo, r.y_hi);
    return r;
}

typedef real real2v __attribute__((ext_vector_type(2)));
typedef real real3v __attribute__((ext_vector_type(3)));
typedef real real4v __attribute__((ext_vector_type(4)));
typedef int int3v __attribute__((ext_vector_type(3)));

// All that the forward pass reads of a triangle, in one piece of 128 bytes (a line of the L2): made by frame_scan_kernel, which has its vertices
// in hand.  (The backward pass reads x and y of the vertices too, from the array, by the record's vertex numbers.)  A list entry's triangle can be anywhere, and by itself its matrix, vertex numbers, vertices, opacities and colours are on
// six or seven lines, each fetched whole for a few bytes and through three loads that wait for each other.
// 10^6 triangles on 1920 x 1080, us, without and with: forward per-pixel order 470, 421 and behind a backward pass, whose gradients
// have taken the caches, 518, 414; tile order 209, 187; backward 911, 880 and 365, 345; the scan 45, 69.  200 000 faint ones, lists of 3700:
// forward 274, 254, backward 203, 196.
// The reach is kept in 16 bits a bound, in fixed steps rounded to the outside: a sixteenth of a pixel of 1920 columns or less everywhere
// (halves, a pixel coarse where the image's edges are: 10^6 triangles, frames, train 1485 -> 1479, shown 591 -> 586).
struct TriangleRecord {
    real4v q[8];  // matrix 0..3 | matrix 4..7 | matrix 8, z | w, reach in x | reach in y, opacities | colours 0..3 | colours 4..7 | colours 8, vertex numbers

    static __device__ __forceinline__ const real4v *at(const RasterArgs &a, int tri) { return reinterpret_cast<const real4v *>(a.records) + 8 * (int64_t)tri; }
    __device__ __forceinline__ void fetch_matrix(const real4v *p) {  // and w, z, the reach
#pragma unroll
        for (int k = 0; k < 4; k++) q[k] = p[k];
        q[4][0] = reinterpret_cast<const real *>(p + 4)[0];
    }
    __device__ __forceinline__ void fetch_attributes(const real4v *p) {  // and the vertex numbers
#pragma unroll
        for (int k = 4; k < 8; k++) q[k] = p[k];
    }
    template <typename R>
    __device__ __forceinline__ void get_matrix(R &r) const {
#pragma unroll
        for (int k = 0; k < 4; k++) { r.m[k] = q[0][k]; r.m[4 + k] = q[1][k]; }
        r.m[8] = q[2][0];
#pragma unroll
        for (int k = 0; k < 3; k++) r.w[k] = q[3][k];
    }
    template <typename R>
    __device__ __forceinline__ void get_attributes(R &r) const {
#pragma unroll
        for (int k = 0; k < 3; k++) r.op[k] = q[4][1 + k];
#pragma unroll
        for (int k = 0; k < 4; k++) { r.col[k] = q[5][k]; r.col[4 + k] = q[6][k]; }
        r.col[8] = q[7][0];
    }
    __device__ __forceinline__ void get_depth(DepthRecord &r) const {
        get_matrix(r);
#pragma unroll
        for (int k = 0; k < 3; k++) r.z[k] = q[2][1 + k];
        r.extent = height();
    }
    __device__ __forceinline__ int3v vertices() const { return int3v{int_of_real((real)q[7][1]), int_of_real((real)q[7][2]), int_of_real((real)q[7][3])}; }

    // Two bounds in steps of 2^-14, rounded away from each other and held in [-2, 2), which no pixel is beyond; NaN leaves nothing out.
    static __device__ __forceinline__ uint32_t pack_bounds(float lo, float hi) {
        constexpr float kStep = 0x1p-14f, kLeast = -2.0f, kMost = 2.0f - kStep;
        const int l = (int)__builtin_floorf(__builtin_fminf(__builtin_fmaxf(lo, kLeast), kMost) / kStep);
        const int h = (int)__builtin_ceilf(__builtin_fmaxf(__builtin_fminf(hi, kMost), kLeast) / kStep);
        return (uint32_t)(uint16_t)l | (uint32_t)h << 16;
    }
    static __device__ __forceinline__ real lower(real packed) { return (real)0x1p-14f * (real)(int16_t)int_of_real(packed); }
    static __device__ __forceinline__ real upper(real packed) { return (real)0x1p-14f * (real)(int16_t)(int_of_real(packed) >> 16); }
    static __device__ __forceinline__ Reach unpack_reach(real x, real y) { return Reach{lower(x), upper(x), lower(y), upper(y)}; }
    __device__ __forceinline__ Reach reach() const { return unpack_reach(q[3][3], q[4][0]); }
    __device__ __forceinline__ real height() const { return upper(q[4][0]) - lower(q[4][0]); }
};

// The matrix of a triangle.  A frame with records has no others.
template <bool kPacked>
__device__ __forceinline__ const real *matrix_of(const RasterArgs &a, int tri) {
    return kPacked ? reinterpret_cast<const real *>(TriangleRecord::at(a, tri)) : a.bary + 9 * (int64_t)tri;
}
// kPacked: from the triangle's record (TriangleRecord), here and below; its reach comes with it.
template <bool kPacked, bool kInHalves = false>
__device__ __forceinline__ Reach gather_blend(const RasterArgs &a, int j, BlendRecord &r) {
    if constexpr (kPacked) {
        const real4v *p = TriangleRecord::at(a, a.sorted_ids[j]);
        TriangleRecord t;
        t.fetch_matrix(p);
        t.get_matrix(r);
        const Reach reach = t.reach();
        r.extent = t.height();
        if (kInHalves) asm volatile("" ::: "memory");  // this half is in LDS before the other one takes its registers
        t.fetch_attributes(p);
        t.get_attributes(r);
#pragma unroll
        for (int k = 0; k < 3; k++) r.iw[k] = 1.0f / r.w[k];
        return reach;
    }
    const TriIds t = load_ids(a, j);
    const real *m = a.bary + 9 * (int64_t)t.tri;
#pragma unroll
    for (int k = 0; k < 9; k++) r.m[k] = m[k];
    const real4 va = a.vertices[t.ia], vb = a.vertices[t.ib], vc = a.vertices[t.ic];
    const real wa = va.w, wb = vb.w, wc = vc.w;
    r.extent = max3(va.y, vb.y, vc.y) - min3(va.y, vb.y, vc.y);
    r.w[0] = wa; r.w[1] = wb; r.w[2] = wc;
    r.iw[0] = 1.0f / wa; r.iw[1] = 1.0f / wb; r.iw[2] = 1.0f / wc;
    gather_attributes(a, t.ia, t.ib, t.ic, r);
    return reaches_everywhere();
}

template <bool kPacked>
__device__ __forceinline__ Reach gather_depth(const RasterArgs &a, int j, DepthRecord &r) {
    if constexpr (kPacked) {
        TriangleRecord t;
        t.fetch_matrix(TriangleRecord::at(a, a.sorted_ids[j]));
        t.get_depth(r);
        return t.reach();
    }
    const TriIds t = load_ids(a, j);
    const real *m = a.bary + 9 * (int64_t)t.tri;
#pragma unroll
    for (int k = 0; k < 9; k++) r.m[k] = m[k];
    const real4 va = a.vertices[t.ia], vb = a.vertices[t.ib], vc = a.vertices[t.ic];
    r.z[0] = va.z; r.z[1] = vb.z; r.z[2] = vc.z;
    r.w[0] = va.w; r.w[1] = vb.w; r.w[2] = vc.w;
    r.extent = max3(va.y, vb.y, vc.y) - min3(va.y, vb.y, vc.y);
    return reaches_everywhere();
}

// A BlendRecord where the triangle's matrix and vertex numbers are known.
template <typename Ids>
__device__ __forceinline__ void gather_record(const RasterArgs &a, const real m[9], const Ids &id, BlendRecord &r) {
#pragma unroll
    for (int k = 0; k < 9; k++) r.m[k] = m[k];
    asm volatile("" ::: "memory");  // the matrix is out of the registers before the rest is asked for
    const real wa = a.vertices[id.x].w, wb = a.vertices[id.y].w, wc = a.vertices[id.z].w;
    r.w[0] = wa; r.w[1] = wb; r.w[2] = wc;
    r.iw[0] = 1.0f / wa; r.iw[1] = 1.0f / wb; r.iw[2] = 1.0f / wc;
    gather_attributes(a, id.x, id.y, id.z, r);
}

// The same from the triangle's record.
__device__ __forceinline__ void gather_record(const RasterArgs &a, const real m[9], int tri, BlendRecord &r) {
    const real4v *p = TriangleRecord::at(a, tri);
    TriangleRecord t;
    t.q[3] = p[3];
    t.fetch_attributes(p);
#pragma unroll
    for (int k = 0; k < 9; k++) r.m[k] = m[k];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        r.w[k] = t.q[3][k];
        r.iw[k] = 1.0f / r.w[k];
    }
    t.get_attributes(r);
}

// gather_depth in steps, for a caller that asks for a record's parts before it needs them.  The parts stay as they were
// loaded (whole vectors, put together by `record` only): a copy into another register would wait for the load.  A vector of
// three is read as the bytes it holds: through a pointer of its own type it would be read as four and from a 16-byte boundary.
struct __attribute__((packed, aligned(4))) Matrix9 { real4v a, b; real c; };
template <typename V, typename T>
__device__ __forceinline__ V read_three(const T *p) {
    V v;
    __builtin_memcpy(&v, p, 3 * sizeof(T));
    return v;
}
struct DepthParts {
    int tri;
    int3v id;
    real4v m0, m1;
    real m2;
    real3v va, vb, vc;  // y, z, w of the vertices

    __device__ __forceinline__ void fetch_triangle(const RasterArgs &a, int j) { tri = a.sorted_ids[j]; }
    // the triangle's vertex numbers and matrix
    __device__ __forceinline__ void fetch_matrix(const RasterArgs &a) {
        const int64_t t = tri;
        id = read_three<int3v>(a.indices + 3 * t);
        const Matrix9 *m = reinterpret_cast<const Matrix9 *>(a.bary + 9 * t);
        m0 = m->a;
        m1 = m->b;
        m2 = m->c;
    }
    __device__ __forceinline__ void fetch_vertices(const RasterArgs &a) {
        const real *v = reinterpret_cast<const real *>(a.vertices) + 1;
        va = read_three<real3v>(v + 4 * (int64_t)id.x);
        vb = read_three<real3v>(v + 4 * (int64_t)id.y);
        vc = read_three<real3v>(v + 4 * (int64_t)id.z);
    }
    __device__ __forceinline__ void get_matrix(real m[9]) const {
#pragma unroll
        for (int k = 0; k < 4; k++) { m[k] = m0[k]; m[4 + k] = m1[k]; }
        m[8] = m2;
    }
    __device__ __forceinline__ DepthRecord record() const {
        DepthRecord r;
        get_matrix(r.m);
        r.z[0] = va[1]; r.z[1] = vb[1]; r.z[2] = vc[1];
        r.w[0] = va[2]; r.w[1] = vb[2]; r.w[2] = vc[2];
        r.extent = max3(va[0], vb[0], vc[0]) - min3(va[0], vb[0], vc[0]);
        return r;
    }
    __device__ __forceinline__ Reach reach(const DepthRecord &) const { return reaches_everywhere(); }
};
// The same with x of the vertices: whole vertices, from 16-byte boundaries in both precisions.
struct __attribute__((packed, aligned(16))) Vertex4 { real4v v; };
struct PlacedParts : DepthParts {
    real4v pa, pb, pc;

    __device__ __forceinline__ void fetch_vertices(const RasterArgs &a) {
        const Vertex4 *v = reinterpret_cast<const Vertex4 *>(a.vertices);
        pa = v[id.x].v;
        pb = v[id.y].v;
        pc = v[id.z].v;
    }
    __device__ __forceinline__ DepthRecord record() const {
        DepthParts d = *this;
        d.va = pa.yzw;
        d.vb = pb.yzw;
        d.vc = pc.yzw;
        return d.record();
    }
    __device__ __forceinline__ Reach reach(const DepthRecord &r) const { return triangle_reach(r.m, pa.x, pa.y, pb.x, pb.y, pc.x, pc.y); }
};

// The same from the triangle's record.
struct PackedParts {
    int tri;
    real4v q0, q1, q2, q3;
    real reach_y;

    __device__ __forceinline__ void fetch_triangle(const RasterArgs &a, int j) { tri = a.sorted_ids[j]; }
    __device__ __forceinline__ void fetch_matrix(const RasterArgs &a) {
        const real4v *p = reinterpret_cast<const real4v *>(a.records) + 8 * (int64_t)tri;
        q0 = p[0];
        q1 = p[1];
        q2 = p[2];
        q3 = p[3];
        reach_y = reinterpret_cast<const real *>(p + 4)[0];
    }
    __device__ __forceinline__ void fetch_vertices(const RasterArgs &) {}
    __device__ __forceinline__ void get_matrix(real m[9]) const {
#pragma unroll
        for (int k = 0; k < 4; k++) { m[k] = q0[k]; m[4 + k] = q1[k]; }
        m[8] = q2[0];
    }
    __device__ __forceinline__ DepthRecord record() const {
        TriangleRecord t;
        t.q[0] = q0;
        t.q[1] = q1;
        t.q[2] = q2;
        t.q[3] = q3;
        t.q[4][0] = reach_y;
        DepthRecord r;
        t.get_depth(r);
        return r;
    }
    __device__ __forceinline__ Reach reach(const DepthRecord &) const { return TriangleRecord::unpack_reach(q3[3], reach_y); }
};

// Saved hit masks (tile order).  The buffer starts with one word per workgroup of the tile launch
// (index hit_mask_head_index()): the largest `last` among the workgroup's pixels, i.e. how much of the
// list the backward pass has to walk, known to it without waiting for its pixels' loads.  Then, from
// word hit_mask_head_words() on, word (chunk * slots + slot) holds, for the pixel in thread slot `slot`
// of its tile, which of 64 consecutive list entries cover it.  The chunks of a tile whose list starts
// at `start` are numbered from start / 64 + tile: consecutive tiles never share a chunk, and
// n_keys / 64 + n_tiles + 1 chunks hold every list.
__device__ __forceinline__ int64_t hit_mask_chunk(int start, int tile, int relative_position) {
    return (int64_t)(start >> 6) + tile + (relative_position >> 6);
}
__device__ __forceinline__ int64_t hit_mask_head_index(int tile) { return (int64_t)tile * gridDim.z + blockIdx.z; }
__device__ __forceinline__ int64_t hit_mask_head_words(int skipped_rows = 0) { return (int64_t)gridDim.x * (gridDim.y - skipped_rows) * gridDim.z; }

// Where the saved blend order of a pixel lies: layer l of the pixel at low[l * stride], and, in tiles whose list holds more
// than kShortList entries, the high half of its list position at high[l * stride].  Two layouts:
//   planes  (max_layers <= TG_MAX_SAVED_LAYERS) one image plane per layer, the high halves in as many planes behind them
//   pool    (any number of layers) where every depth is a number a pixel blends an entry of its tile's list at most once, so
//           a tile with a list of n entries is given n rows of one word per pixel: row `start + l` of the pool is layer l of
//           the tile whose list starts at `start`, and n_keys rows hold every tile's.  Nothing has to be counted or
//           allocated on the device, and what is never blended is never touched.
// A NaN depth breaks that bound: the last candidate of a selection, it ends the order the next one would resume from, and the
// list is blended again and again.  Layers beyond the rows (order_rows) are neither stored nor walked backwards.
struct OrderStore {
    uint16_t *low;      // null: no order saved
    int64_t high;       // words from a low half to its high half; 0: no list is that long
    int pool_pixels;    // pool: words per row (pixels of a tile, whole waves); 0: planes
};
__device__ __forceinline__ int64_t order_stride(const OrderStore &o, const RasterArgs &a) {
    return o.pool_pixels ? o.pool_pixels : (int64_t)a.W * a.H;
}
// Layers of a pixel there is room for; n_entries: length of its tile's list.
__device__ __forceinline__ int order_rows(const OrderStore &o, const RasterArgs &a, int n_entries) {
    return o.pool_pixels ? n_entries : a.max_layers;
}
// t: the pixel's number inside its tile
__device__ __forceinline__ int64_t order_first(const OrderStore &o, const PixelCoord &p, int list_start, int t) {
    return o.pool_pixels ? (int64_t)list_start * o.pool_pixels + t : (p.valid ? p.index : 0);
}

// Batch bounds: word batch_bound_index(start, tile, p) holds, for the tile whose
// list starts at `start`, a lower bound of the per-pixel depth of every entry at
// relative position >= p (p a multiple of kBoundSpan) and < far_start[tile].  From
// far_start on the list holds the entries whose clipped polygon was empty (sort
// key 1e30): they lie at the end of the list whatever their depth, almost never
// cover a pixel, and are always looked at.  Tiles never share a word;
// n_keys / kBoundSpan + n_tiles + 1 words hold every list.
__device__ __forceinline__ int64_t batch_bound_index(int start, int tile, int relative_position) {
    return (int64_t)(start / kBoundSpan) + tile + relative_position / kBoundSpan;
}

// Front-to-back compositing state of one pixel (render.cu:564-574).
struct PixelState {
    real alpha = 1.0f, c0 = 0.0f, c1 = 0.0f, c2 = 0.0f, depth = 0.0f, weight = 0.0f;
    int blended = 0;
};

// The arithmetic of process_forward for a fragment known to be inside.
__device__ __forceinline__ void blend_fragment(PixelState &s, const BlendRecord &r, real b0, real b1, real b2) {
    real o = interp_w(b0, b1, b2, r.op[0], r.op[1], r.op[2], r.w[0], r.w[1], r.w[2]);
    o = clampf(o, 0.0f, kMaxOpacity);
    const real k0 = interp_w(b0, b1, b2, r.col[0], r.col[3], r.col[6], r.w[0], r.w[1], r.w[2]);
    const real k1 = interp_w(b0, b1, b2, r.col[1], r.col[4], r.col[7], r.w[0], r.w[1], r.w[2]);
    const real k2 = interp_w(b0, b1, b2, r.col[2], r.col[5], r.col[8], r.w[0], r.w[1], r.w[2]);
    const real z = interp_1(b0, b1, b2, r.iw[0], r.iw[1], r.iw[2]);
    const real ao = s.alpha * o;
    s.depth = s.depth + ao * z;
    s.weight = s.weight + ao;
    s.c0 = s.c0 + ao * k0;
    s.c1 = s.c1 + ao * k1;
    s.c2 = s.c2 + ao * k2;
    s.alpha *= (1.0f - o);
    s.blended++;
}

// ---- host-side launch helpers (defined in tg_forward.hip) ---------------------------
struct TileLaunch { dim3 grid; int threads; };
TileLaunch tile_launch(int width, int height, int tile_w, int tile_h, int max_threads);
int pixel_order_threads(int preferred);
size_t pixel_order_lds_bytes(int n_threads, int staged_entries, size_t position_bytes = sizeof(int), int places = kLayers);
inline int order_pool_pixels(int tile_w, int tile_h) { return ceil_div(tile_w * tile_h, kWave) * kWave; }
int check_raster_args(const char *fn, int width, int height, int tile_w, int tile_h, int max_layers);

// ---- per-wave culling ------------------------------------------------------------------
// A wave owns 64 pixels of the tile.  Before its lanes test a list entry, the
// entry is tested once against the rectangle spanned by the wave's pixel
// centres.  The test is exact, not approximate: every IEEE operation is monotone
// in each operand, so the inside test's own expression m0*x + m1*y + m2,
// evaluated with the same operations at the corner that maximises it, bounds
// the value every pixel of the rectangle would compute.  If that bound is below
// the inside threshold for one of the three coordinates, no lane can hit.
struct WaveRect { real x_lo, x_hi, y_lo, y_hi; };

__device__ __forceinline__ bool may_touch(const real m[9], const WaveRect &r) {
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const real mx = m[3 * k], my = m[3 * k + 1];
        const real x = (mx >= 0.0f) ? r.x_hi : r.x_lo;
        const real y = (my >= 0.0f) ? r.y_hi : r.y_lo;
        const real bound = mx * x + my * y + m[3 * k + 2];
        if (bound < kEffZero) return false;  // a NaN bound never culls
    }
    return true;
}

__device__ __forceinline__ real min_real(real a, real b) { return (b < a) ? b : a; }
__device__ __forceinline__ real max_real(real a, real b) { return (a < b) ? b : a; }
__device__ __forceinline__ real wave_min(real v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = min_real(v, __shfl_xor(v, off, kWave));
    return v;
}
__device__ __forceinline__ real wave_max(real v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = max_real(v, __shfl_xor(v, off, kWave));
    return v;
}

__device__ __forceinline__ float lane_value(float v, int lane) { return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), lane)); }
__device__ __forceinline__ double lane_value(double v, int lane) {
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const uint64_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, lane), hi = (uint32_t)__builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __longlong_as_double((long long)((hi << 32) | lo));
}

__device__ __forceinline__ real first_value(real v) { return lane_value(v, 0); }  // of a value that is the same in all lanes

constexpr int kMaxTileWaves = kTileThreads / kWave;

// The rectangle of a wave's valid pixels: empty (lo > hi) if it has none.
// Of a square of 8 x 8 it is the coordinates of two lanes: pixel_ndc is monotone, and the pixels that the image does not
// have are the last columns and rows.  (By exchanges between the lanes, 24 round trips through LDS, it was a third of what a wave does
// besides its list.  Forward kernel in per-pixel order, us, with it, the first and the last look whether a tile's pixels want more, and the divisions of
// divide: 10^5 triangles 72, 66, a mesh of 1.3 million 273, 261, 10^6 487, 471.)
__device__ __forceinline__ WaveRect wave_rect(const RasterArgs &a, const PixelCoord &p) {
    const real big = 3.0e38f;
    WaveRect r;
    if (((a.tw | a.th) & 7) == 0) {
        const int columns = a.W - __builtin_amdgcn_readfirstlane(p.ix), rows = a.H - __builtin_amdgcn_readfirstlane(p.iy);
        const bool any = __builtin_amdgcn_readfirstlane((int)p.valid);  // the first lane's, if any
        const int last_column = max(min(columns, 8) - 1, 0), last_row = max(min(rows, 8) - 1, 0);
        r.x_lo = any ? lane_value(p.px, 0) : big;
        r.x_hi = any ? lane_value(p.px, last_column) : -big;
        r.y_lo = any ? lane_value(p.py, 0) : big;
        r.y_hi = any ? lane_value(p.py, 8 * last_row) : -big;
        return r;
    }
    r.x_lo = first_value(wave_min(p.valid ? p.px : big));
    r.x_hi = first_value(wave_max(p.valid ? p.px : -big));
    r.y_lo = first_value(wave_min(p.valid ? p.py : big));
    r.y_hi = first_value(wave_max(p.valid ? p.py : -big));
    return r;
}

// Every wave publishes its rectangle; call with all threads, followed by __syncthreads().
__device__ __forceinline__ void publish_wave_rect(const RasterArgs &a, const PixelCoord &p, WaveRect *s_rects) {
    const WaveRect r = wave_rect(a, p);
    if ((threadIdx.x & (kWave - 1)) == 0) s_rects[threadIdx.x / kWave] = r;
}

// Bit w of the result: wave w has to look at the entry.  The edges' bounds alone let a small triangle reach far past its corners;
// with its reach as well a quarter of the tests go at a mean edge of 4 pixels, four in ten at 1.5.  What finds it is a wave that
// the others wait for, so it is where batches are of 64 entries in per-pixel order, where it gains (forward kernel, us, without
// and with: 10^6 triangles of 4 pixels 596, 575, of 1.5 288, 272, half a million of a mesh 299, 282; 20 000 of 80 pixels 799, 805).  Batches
// of 128 of deep lists lose 1 %, and tile order, whose waves have no registers left for it, gains 2 % from small triangles and
// loses 3 from large ones.
__device__ __forceinline__ uint32_t waves_touched(const real m[9], const WaveRect *s_rects, int n_waves, const Reach &reach = reaches_everywhere()) {
    uint32_t bits = 0;
#pragma unroll 1
    for (int w = 0; w < n_waves; w++) {
        const WaveRect r = s_rects[w];
        const bool beside = r.x_hi < reach.x_lo || r.x_lo > reach.x_hi || r.y_hi < reach.y_lo || r.y_lo > reach.y_hi;  // NaN: not
        if (r.x_lo <= r.x_hi && !beside && may_touch(m, r)) bits |= 1u << w;
    }
    return bits;
}

// 64 staged entries starting at `first`: mask of those the calling wave has to look at.
__device__ __forceinline__ uint64_t wave_candidates(const uint8_t *s_touch, int first, int n_entries, int wave) {
    const int e = first + (threadIdx.x & (kWave - 1));
    const bool mine = e < n_entries && ((s_touch[e] >> wave) & 1u);
    return __builtin_amdgcn_ballot_w64(mine);
}

// Entries whose vertices span less than this many pixel rows are small, and are tested the other way round (lane = entry,
// small_entry_hits) in a tile whose list is long (tests_small_entries), where 64 entries hold at least TG_SMALL_MIN of them.
// That costs about as much as 20 tests by broadcast whatever their number; below it the broadcast wins, and with 10 instead of
// 20 a frame of mixed sizes (10^6 triangles, mean edge 4 pixels) loses 10 % in per-pixel order and 30 % in tile order.  Entries
// of 6 or 12 rows make the tallest lane's rows the whole wave's time (tile order, the same frame: 213 -> 218 -> 249 us).
#ifndef TG_SMALL_ROWS
#define TG_SMALL_ROWS 4.0f
#endif
#ifndef TG_SMALL_MIN
#define TG_SMALL_MIN 20
#endif
constexpr int kSmallMin = TG_SMALL_MIN;
constexpr uint32_t kSmallEntry = 0x80;  // flag in an entry's s_touch byte, next to the waves it touches: to be tested lane by lane
// Whether a tile's small entries are tested lane by lane.  What that gains is the time of a list that the launch waits for,
// alone on its CU with the latency of its LDS reads; a list like all others runs among them on a chip full of instructions,
// and loses.  So: a wave's pixels are a square of 8 x 8, and the frame has no more tiles than CUs (a list of 550 on 64 tiles:
// 47 us with, 65 without), or the list has 1024 entries (5500 on 1024 tiles, tile order: 367 and 529), or 256 and four times
// the mean (650 on 384 tiles with a mean of 85: 60 and 84).  Without the last two conditions, and with them, in tile order: 10^6
// triangles of 1.5 pixels 172 and 140 us, an icosphere of 1.3 million at 1920 x 1080 325 and 270 (three times the mean 283).
constexpr int kFewTiles = 256, kLongSmallList = 1024, kShortSmallList = 256, kSmallListMeans = 4;
__device__ __forceinline__ bool tests_small_entries(const RasterArgs &a, int list_length, int n_tiles) {
    if ((a.tw | a.th) & 7) return false;
    if (n_tiles <= kFewTiles || list_length >= kLongSmallList) return true;
    return list_length >= kShortSmallList && (int64_t)list_length * n_tiles >= (int64_t)kSmallListMeans * a.offsets[n_tiles];
}
__device__ __forceinline__ uint32_t small_entry(const RasterArgs &a, real extent, bool tests_small) {
    return tests_small && extent * (real)a.H < (real)(2.0f * TG_SMALL_ROWS) ? kSmallEntry : 0u;  // NaN: not small
}

// bary_inside in two operations: a minimum passes NaNs by, as the three comparisons there do.
__device__ __forceinline__ bool all_inside(real b0, real b1, real b2) { return !(min_number(b0, b1, b2) < kEffZero); }

template <int kCtrl>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, kCtrl, 0xf, 0xf, true);
}
// A step of transpose_bits: two lanes (their words are `v` and `other`) swap the off-diagonal blocks.
// keep: the bits a lane keeps; turn: how far the other lane's word is rotated to the right.
__device__ __forceinline__ uint32_t exchange_blocks(uint32_t v, uint32_t other, uint32_t keep, uint32_t turn) {
    return (v & keep) | (__builtin_amdgcn_alignbit(other, other, turn) & ~keep);
}
// All ones where bit `bit` of the lane is set: a mask of a step is then one literal and one operation, where a choice between
// two literals is kept in registers by the loop around the call.
__device__ __forceinline__ uint32_t lane_bit_mask(int lane, int bit) { return (uint32_t)__builtin_amdgcn_sbfe(lane, bit, 1); }
// Transposes the 64 x 64 bit matrix whose row i is the word x of lane i: afterwards bit i of lane b's word is what bit b of
// lane i's word was.  Six exchange steps between lanes 32, 16, ... 1 apart, each swapping the off-diagonal blocks of that
// size: the first one is a single v_permlane32_swap, the others one lane move, one rotation and one bit selection per half
// (lane moves in registers; the same steps by __shfl_xor are twelve LDS round trips).
__device__ __forceinline__ uint64_t transpose_bits(uint64_t x, int lane) {
    asm volatile("" : "+v"(lane));  // the masks are made here, not kept by the loop around the call
    const auto halves = __builtin_amdgcn_permlane32_swap((uint32_t)x, (uint32_t)(x >> 32), false, false);
    uint32_t a = halves[0], b = halves[1];
    {
        const auto rows_a = __builtin_amdgcn_permlane16_swap(a, a, false, false), rows_b = __builtin_amdgcn_permlane16_swap(b, b, false, false);
        const bool upper = lane & 16;
        const uint32_t keep = 0x0000FFFFu ^ lane_bit_mask(lane, 4);
        a = exchange_blocks(a, upper ? rows_a[0] : rows_a[1], keep, 16);
        b = exchange_blocks(b, upper ? rows_b[0] : rows_b[1], keep, 16);
    }
    {
        const uint32_t upper = lane_bit_mask(lane, 3), keep = 0x00FF00FFu ^ upper, turn = 24 ^ (upper & 16);  // 24 or 8
        a = exchange_blocks(a, dpp_u32<0x128>(a), keep, turn);  // row_ror:8
        b = exchange_blocks(b, dpp_u32<0x128>(b), keep, turn);
    }
    {
        const uint32_t upper = lane_bit_mask(lane, 2), keep = 0x0F0F0F0Fu ^ upper, turn = 28 ^ (upper & 24);  // 28 or 4
        a = exchange_blocks(a, dpp_u32<0x1B>(dpp_u32<0x141>(a)), keep, turn);  // mirrored inside eight lanes, then inside four
        b = exchange_blocks(b, dpp_u32<0x1B>(dpp_u32<0x141>(b)), keep, turn);
    }
    {
        const uint32_t upper = lane_bit_mask(lane, 1), keep = 0x33333333u ^ upper, turn = 30 ^ (upper & 28);  // 30 or 2
        a = exchange_blocks(a, dpp_u32<0x4E>(a), keep, turn);
        b = exchange_blocks(b, dpp_u32<0x4E>(b), keep, turn);
    }
    {
        const uint32_t upper = lane_bit_mask(lane, 0), keep = 0x55555555u ^ upper, turn = 31 ^ (upper & 30);  // 31 or 1
        a = exchange_blocks(a, dpp_u32<0xB1>(a), keep, turn);
        b = exchange_blocks(b, dpp_u32<0xB1>(b), keep, turn);
    }
    return ((uint64_t)b << 32) | a;
}

// Inside tests the other way round, for 64 entries and a wave that owns a square of 8 x 8 pixels: lane = entry (m: its matrix).
// A lane (mine: its entry is to be tested) first finds the pixel rows its entry can reach, by the same monotone bound as
// may_touch on a strip of one row, and then tests the eight pixels of those rows with the arithmetic of the test itself, so
// the result is that of 64 tests per entry.  -> bit 8 * row + column: the calling lane's entry covers that pixel.
// A test by broadcast costs about 20 vector instructions per entry for all 64 pixels and waits for its LDS reads (200
// clocks where a long list leaves its tile alone on the CU); here 64 entries cost 250 instructions and 110 per row of the
// tallest, all from registers.  500 000 triangles of a mesh, 500 x 500, tile order (longest list 5500 entries): 529 -> 367 us.
// reached_rows reads the coordinates of eight lanes: all lanes of the wave call it, those without an entry leave the result.
__device__ __forceinline__ uint32_t reached_rows(const real m[9], bool mine, const WaveRect &rect, real py) {
    uint32_t rows = 0;
    real mx[3];
#pragma unroll
    for (int k = 0; k < 3; k++) mx[k] = m[3 * k] * (m[3 * k] >= 0.0f ? rect.x_hi : rect.x_lo);
#pragma unroll
    for (int r = 0; r < 8; r++) {
        const real y = lane_value(py, 8 * r);
        const bool reached = all_inside(mx[0] + m[1] * y + m[2], mx[1] + m[4] * y + m[5], mx[2] + m[7] * y + m[8]);
        rows |= reached ? 1u << r : 0u;
    }
    return mine ? rows : 0u;
}
// rows: the pixel rows to test.
__device__ __forceinline__ uint64_t covered_pixels(const real m[9], uint32_t rows, real px, real py) {
    uint64_t covered = 0;
    while (__builtin_amdgcn_ballot_w64(rows != 0)) {  // wave-uniform
        const int r = rows ? __builtin_ctz(rows) : 0;
        const real y = __shfl(py, 8 * r, kWave);
        const real y0 = m[1] * y, y1 = m[4] * y, y2 = m[7] * y;
        uint32_t bits = 0;
#pragma unroll
        for (int c = 0; c < 8; c++) {
            const real x = lane_value(px, c);
            bits |= all_inside(m[0] * x + y0 + m[2], m[3] * x + y1 + m[5], m[6] * x + y2 + m[8]) ? 1u << c : 0u;
        }
        if (rows) covered |= (uint64_t)bits << (8 * r);
        rows &= rows - 1;
    }
    return covered;
}
// The same for the 64 records at s_rec -> bit e: entry e covers the calling lane's pixel.
template <typename Rec>
__device__ __forceinline__ uint64_t small_entry_hits(const Rec *s_rec, bool mine, const WaveRect &rect, real px, real py) {
    const int lane = threadIdx.x & (kWave - 1);
    real m[9];
#pragma unroll
    for (int k = 0; k < 9; k++) m[k] = s_rec[lane].m[k];
    return transpose_bits(covered_pixels(m, reached_rows(m, mine, rect, py), px, py), lane);
}

// The inside tests of 64 entries against a wave's pixels where every lane holds an entry's matrix and nothing is in LDS (mine:
// there is one): 20 or more that can touch the pixels as above, fewer one by one, their matrices read from the lane that has
// them.  -> bit e: entry e covers the calling lane's pixel; hit: the entries that cover any of the pixels.
__device__ __forceinline__ uint64_t wave_hits(const real m[9], bool mine, bool by_lane, const WaveRect &rect, real px, real py,
                                              uint64_t &hit, int lane = threadIdx.x & (kWave - 1)) {
    asm volatile("" : "+v"(lane), "+v"(px), "+v"(py));  // the pixels' coordinates by row and column are made here, not kept by the loop around the call
    const bool candidate = mine && rect.x_lo <= rect.x_hi && may_touch(m, rect);
    uint64_t todo = __builtin_amdgcn_ballot_w64(candidate), hits = 0;
    hit = 0;
    if (by_lane && __builtin_popcountll(todo) >= kSmallMin) {  // wave-uniform
        const uint64_t covered = covered_pixels(m, reached_rows(m, candidate, rect, py), px, py);
        hit = __builtin_amdgcn_ballot_w64(covered != 0);
        return transpose_bits(covered, lane);
    }
    while (todo) {  // wave-uniform
        const int e = __builtin_ctzll(todo);
        todo &= todo - 1;
        real t[9], b0, b1, b2;
#pragma unroll
        for (int k = 0; k < 9; k++) t[k] = lane_value(m[k], e);
        bary_apply(t, px, py, b0, b1, b2);
        const bool inside = all_inside(b0, b1, b2);
        if (inside) hits |= 1ull << e;
        if (__builtin_amdgcn_ballot_w64(inside)) hit |= 1ull << e;
    }
    return hits;
}

// Inside tests of one staged batch for the calling lane's pixel: bit e of the
// result (word e / 64) is set when record e covers the pixel.  Only records that
// can touch the wave's pixels are looked at: all lanes of the wave read the same
// record at the same time (LDS broadcast), or, where 20 or more of 64 entries are
// marked as small, those are tested lane by lane.
// Rec must have a member m[9].
template <int kWords, typename Rec>
__device__ __forceinline__ void batch_hit_mask(const Rec *s_rec, const uint8_t *s_touch, const WaveRect *s_rects, int nb, int wave,
                                               real px, real py, uint64_t m[kWords]) {
#pragma unroll
    for (int wd = 0; wd < kWords; wd++) {
        const int e = wd * kWave + (threadIdx.x & (kWave - 1));
        const uint32_t touch = e < nb ? s_touch[e] : 0u;
        const bool candidate = (touch >> wave) & 1u;
        uint64_t todo = __builtin_amdgcn_ballot_w64(candidate);
        uint64_t hits = 0;
        const bool is_small = candidate && (touch & kSmallEntry);
        const uint64_t small = __builtin_amdgcn_ballot_w64(is_small);
        // wave-uniform; `likely` lays the tests out in line, which long lists in tile order feel (a list of 5500: 382 -> 367 us)
        if (__builtin_expect(__builtin_popcountll(small) >= kSmallMin, 1)) {
            hits = small_entry_hits(s_rec + wd * kWave, is_small, s_rects[wave], px, py);
            todo &= ~small;
        }
        // the lane's mask is built in 32-bit halves: a set bit then costs three vector operations, not six
        uint32_t half[2] = {(uint32_t)hits, (uint32_t)(hits >> 32)};
#pragma unroll
        for (int h = 0; h < 2; h++) {
            uint32_t left = (uint32_t)(todo >> (32 * h));
            while (left) {
                const int bit = __builtin_ctz(left);
                left &= left - 1;
                real b0, b1, b2;
                bary_apply(s_rec[wd * kWave + 32 * h + bit].m, px, py, b0, b1, b2);
                if (all_inside(b0, b1, b2)) half[h] |= 1u << bit;
            }
        }
        m[wd] = ((uint64_t)half[1] << 32) | half[0];
    }
}

__device__ __forceinline__ uint32_t lanes_below_mask(uint64_t mask) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

template <int kWords>
__device__ __forceinline__ bool any_set(const uint64_t m[kWords]) {
    uint64_t all = 0;
#pragma unroll
    for (int wd = 0; wd < kWords; wd++) all |= m[wd];
    return all != 0;
}
// Lowest set bit of a mask of kWords 64-bit words, removed from the mask; -1 if the mask is empty.
template <int kWords>
__device__ __forceinline__ int pop_lowest(uint64_t m[kWords]) {
    int e = -1;
#pragma unroll
    for (int wd = 0; wd < kWords; wd++)
        if (e < 0 && m[wd]) {
            e = 64 * wd + __builtin_ctzll(m[wd]);
            m[wd] &= m[wd] - 1;
        }
    return e;
}

// Per-pixel candidate lists of the per-pixel-sort mode live in LDS, slot-major:
// entry `slot` of thread `t` is at [slot * n_threads + t] (conflict-free).
template <typename Pos>
struct TopKOf {
    real *depth;
    Pos *pos;
    int n_threads;
    __device__ __forceinline__ real &d(int slot) const { return depth[slot * n_threads + threadIdx.x]; }
    __device__ __forceinline__ Pos &j(int slot) const { return pos[slot * n_threads + threadIdx.x]; }
};
using TopK = TopKOf<int>;

}  // namespace tg
