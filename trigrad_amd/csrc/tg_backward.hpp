// tg_backward.hpp -- backward kernels of the tile compositor, a wave to 64 pixels of a tile.  (Launched in tg_backward.hip; the instances
// that read triangles' records are compiled in tg_backward_packed.hip.)
//
// Fragments are visited in exact reverse blend order; the transmittance in front
// of a fragment is reconstructed by dividing the running value by (1 - opacity),
// as the reference does (render.cu:492).
//
// Each fragment yields 21 gradient terms (3 vertices x {x, y, w, r, g, b,
// opacity}; the z gradient is identically zero, render.cu:531-533).  Terms of
// the same list entry are added up inside a wave before they reach memory, so
// the kernels issue one global floating-point atomic per (wave, run of equal
// entries, term) instead of 24 per (pixel, entry).
//
// per_pixel_sort = 0 (backward_tile_order_kernel): all pixels of a tile share
//   the list order, so every wave walks its tile's list backwards in blocks
//   of 64 entries.
// per_pixel_sort = 1 (backward_saved_order_kernel): every
//   pixel walks the blend order the forward pass saved for it, backwards.
// per_pixel_sort = 1, no saved order (backward_pixel_order_kernel): the pixel
//   re-selects its fragments from the far end (32 at a time, below the (depth,
//   position) of the last blended fragment saved by the forward pass).
#pragma once
#include "tg_frame.hpp"
#include "tg_raster.hpp"

namespace tg {

struct BackwardArgs {
    const real4 *grad_image;
    const real *grad_depthmap;
    const real4 *image;
    const real *depthmap;
    const real *weights;
    const int32_t *ends;
    const int32_t *last;
    const real *last_depth;
    OrderStore order;          // the blend order saved by the forward pass
    const uint64_t *hit_masks; // saved by the tile-order forward pass, or null
    real *grad_vertices;
    real *grad_colors;
    real *grad_opacities;
    int vertex_stride, color_stride, opacity_stride;  // scalars from one vertex to the next in the three arrays
    const uint32_t *list_status;  // status word of the kernels that made the lists (TG_STATUS_*); may be null
    int mask_parts, mask_threads; // of the saved hit masks: workgroups of a tile in the forward launch, and their threads
    int64_t copy_stride;          // scalars from one XCD's gradient arrays to the next one's; 0: all XCDs share them
    bool deep;                    // many layers and long lists: which tiles an XCD takes (tile_of_workgroup)
};

// Lists whose sort gave up a wait are not to be read; the host finds the word and raises.
__device__ __forceinline__ bool lists_invalid(const BackwardArgs &g) { return g.list_status && *g.list_status != TG_STATUS_OK; }

// Most losses are of the image alone: kDepth = false is for a frame whose depth map has no gradient.  Its terms by way of the depth
// are then zeros, a sixth of a fragment's arithmetic, and are left out, but for the cases where they are 0 times infinity: the
// NaNs that make of a gradient are kept (depth_is_ordinary, load_back_state).  One kind is not: where the depth's derivative by an
// opacity (fragment_seed) overflows although the pixel's depth is finite, which takes a depth beyond 1e34 or one
// beyond 1e38 times its fragment's opacity, the gradients of that fragment are what the image alone makes them.  The saved-order
// kernel then needs 96 registers, not 117, and five waves a SIMD find room: 10^6 triangles 1219 -> 1043 us, 20 000 without a limit on the
// layers 604 -> 541; in tile order 619 -> 594.

// process_backward's inputs for one list entry.
template <bool kDepth>
struct VertexDepths {
    real iw[3];
    real iw2[3];  // 1 / (w * w)
};
template <>
struct VertexDepths<false> {};
template <bool kDepth>
struct alignas(16) BackRecord : VertexDepths<kDepth> {
    real m[9];
    real w[3];
    real op[3];
    real col[9];
    real xy[6];   // ax, ay, bx, by, cx, cy
    int id[3];
};

// Whether any lane of the wave meets a case that has to be put right (wave-uniform; laid out as the exception).
__device__ __forceinline__ bool any_lane(bool x) { return __builtin_expect(__builtin_amdgcn_ballot_w64(x) != 0, 0); }

// 1 / x to within one unit in the last place: the hardware estimate and one Newton step where
// the estimate is an ordinary number (zero, infinity and NaN pass through as they are).  Used
// where the reference divides in its backward pass and the quotient is no carried state.
__device__ __forceinline__ float reciprocal(float x) {
    const float r = __builtin_amdgcn_rcpf(x);
    const float refined = __builtin_fmaf(__builtin_fmaf(-x, r, 1.0f), r, r);
    return __builtin_amdgcn_classf(r, 0x198) ? refined : r;  // +-normal, +-denormal
}
__device__ __forceinline__ double reciprocal(double x) { return 1.0 / x; }
__device__ __forceinline__ float reciprocal_of_normal(float x) {
    const float r = __builtin_amdgcn_rcpf(x);
    return __builtin_fmaf(__builtin_fmaf(-x, r, 1.0f), r, r);
}
__device__ __forceinline__ double reciprocal_of_normal(double x) { return 1.0 / x; }
// x / y, correctly rounded, for y in [1e-4, 1] and r = reciprocal(y): the quotient x * r put right by its exact remainder twice, the
// steps of the division itself without its scaling (one of them leaves a few operand pairs in millions a unit off).  The
// remainder is a number of float32 as long as x is above 2^-102; other x, which a pixel's transmittance is with a threshold of 0
// only, are divided, with the lanes beside them.  (A branch of the wave, not of the lane, which cost the saved-order kernel 1 %, 10^6
// triangles 1239 us, so 1218; scaled by div_fmas without a branch 1234.  Not expected, and said so here and not in a function
// around the condition, because else the division is made in every case: 1238.  One test for the whole walk, of the
// smallest transmittance at its start, is three operations a fragment less and slower: 1003, 1028.)
__device__ __forceinline__ float quotient(float x, float y, float r) {
    const bool ordinary = __float_as_uint(x) - 0x0d800000u < 0x7f000000u - 0x0d800000u;  // 2^-100 <= x < 2^127
    float q = x * r;
    q = __builtin_fmaf(__builtin_fmaf(-y, q, x), r, q);
    q = __builtin_fmaf(__builtin_fmaf(-y, q, x), r, q);
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(!ordinary) != 0, 0)) q = x / y;
    return q;
}
__device__ __forceinline__ double quotient(double x, double y, double) { return x / y; }

// gradients only: 1 / w to within one unit in the last place, and its square for 1 / (w * w)
__device__ __forceinline__ void vertex_depths(const real w[3], VertexDepths<true> &r) {
#pragma unroll
    for (int k = 0; k < 3; k++) {
        r.iw[k] = reciprocal(w[k]);
        r.iw2[k] = r.iw[k] * r.iw[k];
    }
}

template <bool kDepth>
__device__ __forceinline__ void gather_back(const RasterArgs &a, const TriIds &t, BackRecord<kDepth> &r) {
    const real *m = a.bary + 9 * (int64_t)t.tri;
    real4v va = *reinterpret_cast<const real4v *>(a.vertices + t.ia), vb = *reinterpret_cast<const real4v *>(a.vertices + t.ib),
           vc = *reinterpret_cast<const real4v *>(a.vertices + t.ic);
#pragma unroll
    for (int k = 0; k < 9; k++) r.m[k] = m[k];
    r.op[0] = a.opacities[t.ia]; r.op[1] = a.opacities[t.ib]; r.op[2] = a.opacities[t.ic];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        r.col[k] = a.colors[3 * (int64_t)t.ia + k];
        r.col[3 + k] = a.colors[3 * (int64_t)t.ib + k];
        r.col[6 + k] = a.colors[3 * (int64_t)t.ic + k];
    }
    // z is not used, and without this a vertex would be two loads, x and y, and w (14 instead of 17 loads an entry: 1 % of the
    // saved-order kernel); here, behind all loads, because it is where they are waited for
    asm("" : "+v"(va), "+v"(vb), "+v"(vc));
    r.w[0] = va[3]; r.w[1] = vb[3]; r.w[2] = vc[3];
    if constexpr (kDepth) vertex_depths(r.w, r);
    r.xy[0] = va[0]; r.xy[1] = va[1]; r.xy[2] = vb[0]; r.xy[3] = vb[1]; r.xy[4] = vc[0]; r.xy[5] = vc[1];
    r.id[0] = t.ia; r.id[1] = t.ib; r.id[2] = t.ic;
}
// The same from the triangle's record; of the vertices themselves x and y.
template <bool kDepth>
__device__ __forceinline__ void gather_packed(const RasterArgs &a, int tri, BackRecord<kDepth> &r) {
    TriangleRecord t;
    t.fetch_matrix(TriangleRecord::at(a, tri));
    t.fetch_attributes(TriangleRecord::at(a, tri));
    const int3v id = t.vertices();
    const real2v *v = reinterpret_cast<const real2v *>(a.vertices);
    const real2v va = v[2 * (int64_t)id.x], vb = v[2 * (int64_t)id.y], vc = v[2 * (int64_t)id.z];
    t.get_matrix(r);
    t.get_attributes(r);
    r.id[0] = id.x; r.id[1] = id.y; r.id[2] = id.z;
    if constexpr (kDepth) vertex_depths(r.w, r);
    r.xy[0] = va[0]; r.xy[1] = va[1]; r.xy[2] = vb[0]; r.xy[3] = vb[1]; r.xy[4] = vc[0]; r.xy[5] = vc[1];
}


// Reverse-traversal state of one pixel (render.cu:647-653): what a fragment changes, and what it reads only.
struct ChainState {
    real alpha, s0, s1, s2, oa, zoa;  // oa, zoa: with kDepth
};
struct BackState : ChainState {
    real final_alpha, final_weight, final_depth;
    real inv_final_weight;  // the reference divides two terms of every fragment by the pixel's final weight
    real g0, g1, g2, g3, gd;  // upstream gradient of this pixel
};

constexpr int kTerms = 21;  // per vertex v: [7v+0] x, [7v+1] y, [7v+2] w, [7v+3..5] rgb, [7v+6] opacity

// util.h:299-317 scalar interpolate3_backward.  -> the reference returns early there (util.h:303) and all results are zero: the
// caller's to set, once for all of a fragment's and in a branch that a wave rarely takes.  (A selection at every result is a branch
// around its arithmetic, twelve a fragment: the compiler does not move arithmetic across them.)
__device__ __forceinline__ bool interp_backward_scalar(real g, const real b[3], const real v[3], const real w[3],
                                                       real gb[3], real gv[3], real gw[3]) {
    const real nom = (b[0] * w[0] * v[0] + b[1] * w[1] * v[1]) + b[2] * w[2] * v[2];
    const real denom = (b[0] * w[0] + b[1] * w[1]) + b[2] * w[2];
    const real inv = reciprocal(denom);  // the reference divides nine times, by denom and by its square
    const real inv2 = inv * inv;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        gb[k] = g * ((v[k] * w[k] * denom - nom * w[k]) * inv2);
        gv[k] = g * b[k] * w[k] * inv;
        gw[k] = g * (b[k] * v[k] * denom - nom * b[k]) * inv2;  // g * inv2 overflows where w is around 1e-18
    }
    return denom * denom < kEffZero;
}

// process_backward (render.cu:455-538) is evaluated in two parts.  The part that
// carries state from one fragment of a pixel to the next (transmittance and the
// running sums) has to follow the reverse blend order of that pixel; it reduces
// the fragment to five numbers.  Everything else is a function of those five
// numbers, the pixel position and the triangle, and can be evaluated in any
// order.

// What the ordered part hands over for one fragment.
struct FragSeed {
    real d_do;    // derivative w.r.t. the interpolated opacity (:502)
    real gc[3];   // derivative w.r.t. the interpolated colour (:510)
    real dd_dz;   // derivative w.r.t. the interpolated view depth (:517); with kDepth
};

// The fragment itself: interpolated opacity, colour and, with kDepth, view depth (no state involved).
struct FragValue {
    real o, color[3], z;
};

template <bool kDepth>
__device__ __forceinline__ FragValue fragment_value(const BackRecord<kDepth> &r, real b0, real b1, real b2) {
    const real w[3] = {r.w[0], r.w[1], r.w[2]};
    FragValue v;
    // The opacity is recomputed exactly as the forward pass computed it: 1 - o can be small, and the
    // transmittance is reconstructed by dividing by it.  The three colour quotients over the same
    // denominator (util.h:245-250) share its reciprocal.
    v.o = clampf(interp_w(b0, b1, b2, r.op[0], r.op[1], r.op[2], w[0], w[1], w[2]), 0.0f, kMaxOpacity);
    const real inv_denom = reciprocal(b0 * w[0] + b1 * w[1] + b2 * w[2]);
#pragma unroll
    for (int k = 0; k < 3; k++)
        v.color[k] = (b0 * r.col[k] * w[0] + b1 * r.col[3 + k] * w[1] + b2 * r.col[6 + k] * w[2]) * inv_denom;
    if constexpr (kDepth) v.z = interp_1(b0, b1, b2, r.iw[0], r.iw[1], r.iw[2]);
    return v;
}

// The state behind a fragment, in reverse blend order (render.cu:487-497), from the one in front of it.  om = 1 - o.
template <bool kDepth>
__device__ __forceinline__ ChainState chain_behind(const ChainState &st, const FragValue &v, real om, real inv_om) {
    ChainState next;
    next.alpha = quotient(st.alpha, om, inv_om);                                           // :492 (state: kept exact)
    next.s0 = st.s0 + v.color[0] * v.o * next.alpha;                                       // :493
    next.s1 = st.s1 + v.color[1] * v.o * next.alpha;
    next.s2 = st.s2 + v.color[2] * v.o * next.alpha;
    if constexpr (kDepth) {
        next.oa = st.oa + v.o * next.alpha;                                                // :496
        next.zoa = st.zoa + v.z * v.o * next.alpha;                                        // :497
    }
    return next;
}
// What a fragment's gradient terms are linear in (render.cu:487-517), from the states in front of it and behind it.
template <bool kDepth>
__device__ __forceinline__ FragSeed fragment_seed(const ChainState &st, const ChainState &next, const FragValue &v, real inv_om, const BackState &pixel) {
    const real g[3] = {pixel.g0, pixel.g1, pixel.g2}, s[3] = {st.s0, st.s1, st.s2};
    real t3[3];
#pragma unroll
    for (int k = 0; k < 3; k++) t3[k] = (v.color[k] * st.alpha - s[k]) * inv_om * g[k];
    FragSeed f;
    f.d_do = ((t3[0] + t3[1]) + t3[2]) + pixel.g3 * (-pixel.final_alpha * inv_om);         // :491
    const real ao = next.alpha * v.o;
    f.gc[0] = ao * g[0]; f.gc[1] = ao * g[1]; f.gc[2] = ao * g[2];                         // :510
    if constexpr (kDepth) {
        const real ddw_do = next.alpha - st.oa * inv_om;                                      // :494
        const real dud_do = next.alpha * v.z - st.zoa * inv_om;                               // :495
        real dd_do = (dud_do - pixel.final_depth * ddw_do) * pixel.inv_final_weight * pixel.gd;  // :499
        if (pixel.final_weight < kEffZero) dd_do = 0.0f;
        f.d_do = f.d_do + dd_do;
        f.dd_dz = ao * pixel.gd * pixel.inv_final_weight;                                    // :517
        if (pixel.final_weight < kEffZero) f.dd_dz = 0.0f;
    }
    return f;
}
// 1 - o and its reciprocal; in [1e-4, 1] or NaN; the reference divides six derivative terms by it
struct Remainder { real om, inv; };
__device__ __forceinline__ Remainder remainder_of(real o) {
    const real om = 1.0f - o;
    return {om, reciprocal_of_normal(om)};
}

// Without a gradient of the depth: whether the terms by way of it are zeros.  They are where no product in them can be too large
// for a float.  The coordinates b are positive, so with w and denom = b0 w0 + b1 w1 + b2 w2 in [1e-6, 1e6] the sum of the b
// is in [1e-12, 1e12], and every factor that a zero meets below 1e31.  (A NaN in w or b makes NaNs of all terms without these.)
__device__ __forceinline__ bool depth_is_ordinary(const real w[3], real denom) {
    const real low = 1e-6f, high = 1e6f;
    return min_number(w[0], w[1], w[2]) > low && max_number(w[0], w[1], w[2]) < high && denom > low && denom < high;
}

// The order-free part: the 21 gradient terms of one fragment.
template <bool kDepth>
__device__ __forceinline__ void fragment_terms(const FragSeed &f, const BackRecord<kDepth> &r, real b0, real b1, real b2, real px,
                                               real py, real out[kTerms]) {
    const real b[3] = {b0, b1, b2};
    const real w[3] = {r.w[0], r.w[1], r.w[2]};
    const real ones[3] = {1.0f, 1.0f, 1.0f};
    real gb_o[3], gv_o[3], gw_o[3];
    const bool dead = interp_backward_scalar(f.d_do, b, r.op, w, gb_o, gv_o, gw_o);

    // vector interpolate3_backward for the colour (util.h:319-355)
    const real *gc = f.gc;
    real gb_c[3], gw_c[3], scale[3];
    {
        real nom[3];
#pragma unroll
        for (int k = 0; k < 3; k++) nom[k] = (b[0] * w[0] * r.col[k] + b[1] * w[1] * r.col[3 + k]) + b[2] * w[2] * r.col[6 + k];
        const real denom = b[0] * w[0] + b[1] * w[1] + b[2] * w[2];
        const real inv = reciprocal(denom);
        const real inv2 = inv * inv;
#pragma unroll
        for (int v = 0; v < 3; v++) {
            real dfb[3], dfw[3];
#pragma unroll
            for (int k = 0; k < 3; k++) {
                const real a = r.col[3 * v + k];
                dfb[k] = w[v] * (a * denom - nom[k]) * inv2;
                dfw[k] = b[v] * a * denom - nom[k] * b[v];
            }
            gb_c[v] = (gc[0] * dfb[0] + gc[1] * dfb[1]) + gc[2] * dfb[2];
            gw_c[v] = ((gc[0] * dfw[0] + gc[1] * dfw[1]) + gc[2] * dfw[2]) * inv2;
            scale[v] = b[v] * w[v] * inv;
        }
    }

    real gb_z[3], gv_z[3], gw_z[3];
    bool dead_z = false;
    if constexpr (kDepth) dead_z = interp_backward_scalar(f.dd_dz, b, r.iw, ones, gb_z, gv_z, gw_z);
    if (any_lane(dead || dead_z)) {
#pragma unroll
        for (int k = 0; k < 3; k++) {
            if (dead) gb_o[k] = gv_o[k] = gw_o[k] = gb_c[k] = gw_c[k] = scale[k] = 0.0f;  // util.h:303, :326: the same denominator
            if (dead_z) gb_z[k] = gv_z[k] = gw_z[k] = 0.0f;
        }
    }
    real gbary[3], dw[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        gbary[k] = gb_o[k] + gb_c[k];  // :527
        dw[k] = gw_o[k] + gw_c[k];     // :530
    }
    const auto add_depth = [&](int k, real iw2) {
        gbary[k] += gb_z[k];
        dw[k] = dw[k] + gw_z[k] + -gv_z[k] * iw2;  // :523-525
    };
    if constexpr (kDepth) {
#pragma unroll
        for (int k = 0; k < 3; k++) add_depth(k, r.iw2[k]);
    } else if (any_lane(!depth_is_ordinary(r.w, (b[0] * w[0] + b[1] * w[1]) + b[2] * w[2]))) {
        VertexDepths<true> depths;
        vertex_depths(r.w, depths);
        dead_z = interp_backward_scalar(0.0f, b, depths.iw, ones, gb_z, gv_z, gw_z);
#pragma unroll
        for (int k = 0; k < 3; k++) {
            if (dead_z) gb_z[k] = gv_z[k] = gw_z[k] = 0.0f;
            add_depth(k, depths.iw2[k]);
        }
    }

    // util.h:405-455 barycentric_backward (vertex part)
    const real ax = r.xy[0], ay = r.xy[1], bx = r.xy[2], by = r.xy[3], cx = r.xy[4], cy = r.xy[5];
    real dxy[3][2];
    {
        // The reference divides each of the 21 numerators below by T or d (util.h:405-455).  Here the two
        // reciprocals are formed once: T's is multiplied into l0..l2, each within two units in the last place of
        // the reference's quotient, and d's into the six sums of three products, whose 18 quotients are not formed
        // (19 of the fragment's 50 divisions go away).  The numerators keep the reference's form: its differences of screen coordinates cancel, and for a sliver that rounding
        // is larger than the tolerance of the comparison, so the shorter closed form
        // (-l_v * row k of the matrix) does not reproduce the reference's numbers.
        // Nor are they fused: a fused multiply-add moves l0..l2 by as much as the reference's own rounding
        // does, which the numerators amplify for a sliver (measured: 11 rounding steps of the terms' magnitudes
        // where 2 are allowed), and the same holds for v * denom - nom in interp_backward_scalar (2.6 steps).
        const real T = (bx - ax) * (cy - ay) - (by - ay) * (cx - ax);
        const real inv_T = reciprocal(T);
        const real l0 = ((bx - px) * (cy - py) - (by - py) * (cx - px)) * inv_T;
        const real l1 = ((cx - px) * (ay - py) - (cy - py) * (ax - px)) * inv_T;
        const real l2 = ((ax - px) * (by - py) - (ay - py) * (bx - px)) * inv_T;
        const real d = ax * (by - cy) + bx * (-ay + cy) + cx * (ay - by);
        {
            const real inv_d = reciprocal(d);  // of the sum, not of its 18 numerators: 12 multiplications and as many roundings less
            real J[3][2][3];
            J[0][0][0] = l0 * (-by + cy);
            J[0][0][1] = -cy - l1 * (by - cy) + py;
            J[0][0][2] = by - l2 * (by - cy) - py;
            J[0][1][0] = l0 * (bx - cx);
            J[0][1][1] = cx + l1 * (bx - cx) - px;
            J[0][1][2] = -bx + l2 * (bx - cx) + px;
            J[1][0][0] = cy + l0 * (ay - cy) - py;
            J[1][0][1] = l1 * (ay - cy);
            J[1][0][2] = -ay + l2 * (ay - cy) + py;
            J[1][1][0] = -cx - l0 * (ax - cx) + px;
            J[1][1][1] = l1 * (-ax + cx);
            J[1][1][2] = ax - l2 * (ax - cx) - px;
            J[2][0][0] = -by - l0 * (ay - by) + py;
            J[2][0][1] = ay - l1 * (ay - by) - py;
            J[2][0][2] = l2 * (-ay + by);
            J[2][1][0] = bx + l0 * (ax - bx) - px;
            J[2][1][1] = -ax + l1 * (ax - bx) + px;
            J[2][1][2] = l2 * (ax - bx);
#pragma unroll
            for (int v = 0; v < 3; v++)
#pragma unroll
                for (int c = 0; c < 2; c++)
                    dxy[v][c] = (gbary[0] * J[v][c][0] + gbary[1] * J[v][c][1] + gbary[2] * J[v][c][2]) * inv_d;
            const bool flat = abs_real(d) < kEffZero;  // util.h:421: zero
            if (any_lane(flat)) {
#pragma unroll
                for (int v = 0; v < 3; v++)
                    if (flat) dxy[v][0] = dxy[v][1] = 0.0f;
            }
        }
    }
#pragma unroll
    for (int v = 0; v < 3; v++) {
        out[7 * v + 0] = dxy[v][0];
        out[7 * v + 1] = dxy[v][1];
        out[7 * v + 2] = dw[v];
        out[7 * v + 3] = gc[0] * scale[v];
        out[7 * v + 4] = gc[1] * scale[v];
        out[7 * v + 5] = gc[2] * scale[v];
        out[7 * v + 6] = gv_o[v];
    }
}

// One fragment start to finish (used where every pixel has its own order).
__device__ __forceinline__ void fragment_backward(BackState &st, const BackRecord<true> &r, real b0, real b1, real b2, real px,
                                                  real py, real out[kTerms]) {
    const FragValue v = fragment_value(r, b0, b1, b2);
    const Remainder rem = remainder_of(v.o);
    const ChainState next = chain_behind<true>(st, v, rem.om, rem.inv);
    const FragSeed f = fragment_seed<true>(st, next, v, rem.inv, st);
    static_cast<ChainState &>(st) = next;
    fragment_terms(f, r, b0, b1, b2, px, py, out);
}

// Layout of the three gradient arrays, a template parameter of the kernels so that the two layouts
// in use address with constants: dense (4, 3, 1 scalars per vertex), one (V,8) block (8, 8, 8), or
// the strides given at run time.
enum GradLayout { kGradDense = 0, kGradBlock8 = 1, kGradStrided = 2 };

template <int kLayout>
__device__ __forceinline__ int term_stride(const BackwardArgs &g, int c) {
    if (c < 3) return kLayout == kGradDense ? 4 : kLayout == kGradBlock8 ? 8 : g.vertex_stride;
    if (c < 6) return kLayout == kGradDense ? 3 : kLayout == kGradBlock8 ? 8 : g.color_stride;
    return kLayout == kGradDense ? 1 : kLayout == kGradBlock8 ? 8 : g.opacity_stride;
}

template <int kLayout>
__device__ __forceinline__ real *term_address(const BackwardArgs &g, int vertex_id, int c) {
    const int64_t at = term_stride<kLayout>(g, c) * (int64_t)vertex_id;
    if (c < 2) return g.grad_vertices + at + c;
    if (c == 2) return g.grad_vertices + at + 3;
    if (c < 6) return g.grad_colors + at + (c - 3);
    return g.grad_opacities + at;
}

template <bool kDepth>
__device__ __forceinline__ BackState load_back_state(const BackwardArgs &g, int pixel) {
    BackState st;
    const real4 gi = g.grad_image[pixel];
    st.g0 = gi.x; st.g1 = gi.y; st.g2 = gi.z; st.g3 = gi.w;
    st.gd = g.grad_depthmap ? g.grad_depthmap[pixel] : 0.0f;  // null: the depth map took no part in the loss
    st.final_alpha = g.image[pixel].w;
    st.alpha = st.final_alpha;
    st.s0 = st.s1 = st.s2 = 0.0f;
    st.oa = st.zoa = 0.0f;
    st.final_weight = g.weights[pixel];
    st.inv_final_weight = 1.0f / st.final_weight;
    st.final_depth = g.depthmap[pixel];
    // without a gradient of the depth its part of d_do is 0 times these, and g3 is a factor of d_do only
    if (!kDepth && !(st.final_weight < kEffZero)) st.g3 += st.final_depth * 0.0f + st.inv_final_weight * 0.0f;
    return st;
}


constexpr int kBackBatch = 64;    // list entries of a block, a word of a lane's hit mask
constexpr int kWaveSlots = 64;    // hit slots per wave and round: one per lane of the order-free part
constexpr int kTermStride = 65;   // row stride of the per-wave term matrix (odd: conflict-free columns)
constexpr int kMaxWaves = kTileThreads / kWave;

// The number of the XCD that runs the calling wave.  What depends on it is where sums are kept, not what they are.
__device__ __forceinline__ int xcd_number() {
    constexpr int kXccId = 20, kBits = 4;  // the hardware register and its width
    return (int)__builtin_amdgcn_s_getreg(kXccId | (kBits - 1) << 11) & (kXcds - 1);
}

// The run sums' view of a lane: lane = 21 * group + q adds up gradient term q over the group's third
// of the slots.  What depends on q only is worked out once per kernel.
struct TermLane {
    int group;   // 0..2; 3 for the one lane left over
    int q;
    int vertex;  // q / 7: which of the entry's three vertices the term belongs to
    int stride;  // scalars per vertex in the term's array
    real *base;  // the term's element of vertex 0
};

template <int kLayout>
__device__ __forceinline__ TermLane term_lane(const BackwardArgs &g, int lane) {
    TermLane t;
    t.group = lane / kTerms;
    t.q = lane - t.group * kTerms;
    t.vertex = t.q / 7;
    const int c = t.q - 7 * t.vertex;
    t.stride = term_stride<kLayout>(g, c);
    t.base = term_address<kLayout>(g, 0, c) + g.copy_stride * xcd_number();
    return t;
}

// Adds up the runs of equal list entry among the first n slots of a wave's term matrix (row q = term
// q, rows kTermStride apart; slots of one entry are neighbours) and adds every non-zero run sum to the
// gradient arrays.  Bit c of `heads` is set where slot c starts a run.  Lane (group, q) owns a fixed third of
// row q -- slots [0, 21), [21, 42) or [42, 64) -- and turns it into running sums that start over at each head:
// straight-line code, no branch, no look at the entries; slots from n on hold what an earlier round left, which
// a running sum carries to later slots only, never into a slot below n.  The last slot of a run, and of a third,
// then holds a sum to deliver, and every lane walks the ones of its own third.  vertex_at(c, v): vertex id v of
// the entry in slot c.
// (21, 21 and 22 and not the other way round: the 63 lanes' elements, in banks q + c0 + k, are then 63 banks.)
constexpr int kRunSpan = 21, kLastSpan = kWave - 2 * kRunSpan;
// Bit k of x as a mask, all ones or 0.  (The compiler is not to know that: it makes a comparison and a selection of a mask, three
// operations and a wait for one.)
__device__ __forceinline__ int bit_mask(int x, int k) {
    int mask = __builtin_amdgcn_sbfe(x, k, 1);
    asm("" : "+v"(mask));
    return mask;
}
// x where mask is all ones, 0 where it is 0.
__device__ __forceinline__ float masked(float x, int mask) { return __int_as_float(__float_as_int(x) & mask); }
__device__ __forceinline__ double masked(double x, int mask) { return mask ? x : 0.0; }
template <typename VertexAt>
__device__ __forceinline__ void add_run_sums(real *terms, int n, uint64_t heads, const TermLane &t, VertexAt vertex_at) {
    if (t.group >= 3) return;  // the one lane left over; nothing below synchronises the wave
    const int c0 = t.group * kRunSpan;
    real *row = terms + t.q * kTermStride + c0;
    const bool last = t.group == 2;  // the third of kLastSpan slots
    {
        const int carries = (int)~(uint32_t)(heads >> c0);  // bit k: slot k goes on with the run of the slot before it
        real v[kLastSpan];
#pragma unroll
        for (int k = 0; k < kLastSpan; k++) v[k] = (k < kRunSpan || last) ? row[k] : 0.0f;
        real sum = 0.0f;
#pragma unroll
        for (int k = 0; k < kLastSpan; k++) {
            sum = v[k] + masked(sum, bit_mask(carries, k));
            if (k < kRunSpan || last) row[k] = sum;
        }
    }
    // what a lane reads below it wrote itself above: LDS serves a wave's instructions in order
    uint64_t tails = (heads >> 1) | (1ull << (n - 1)) | (1ull << (kRunSpan - 1)) | (1ull << (2 * kRunSpan - 1));
    if (n < kWave) tails &= (1ull << n) - 1;
    uint32_t mine = (uint32_t)(tails >> c0) & ((1u << (last ? kLastSpan : kRunSpan)) - 1);
    while (mine) {
        // two slots per turn, so that two chains of LDS reads are in flight
        const int k0 = __builtin_ctz(mine);
        mine &= mine - 1;
        const int k1 = mine ? __builtin_ctz(mine) : k0;
        const bool two = mine != 0;
        mine &= mine - 1;  // 0 & anything = 0
        const real sum0 = row[k0], sum1 = two ? row[k1] : 0.0f;
        const int vertex0 = vertex_at(c0 + k0, t.vertex), vertex1 = vertex_at(c0 + k1, t.vertex);
        if (sum0 != 0.0f) unsafeAtomicAdd(t.base + (int64_t)t.stride * vertex0, sum0);
        if (sum1 != 0.0f) unsafeAtomicAdd(t.base + (int64_t)t.stride * vertex1, sum1);
    }
}

__device__ __forceinline__ int top_bit(uint64_t m) { return 63 - __builtin_clzll(m); }

// The largest of the wave's values that are not negative (all lanes must be active; 0 where all are negative): six operations,
// where exchanges by LDS are six round trips, one after the other.
template <int kCtrl, int kRowMask>
__device__ __forceinline__ int dpp_max_i32(int v) {
    return max(v, __builtin_amdgcn_update_dpp(0, v, kCtrl, kRowMask, 0xf, false));
}
__device__ __forceinline__ int wave_max_i32(int v) {
    v = dpp_max_i32<0x111, 0xf>(v);  // row_shr:1, 2, 4, 8
    v = dpp_max_i32<0x112, 0xf>(v);
    v = dpp_max_i32<0x114, 0xf>(v);
    v = dpp_max_i32<0x118, 0xf>(v);
    v = dpp_max_i32<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
    v = dpp_max_i32<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
    return __builtin_amdgcn_readlane(v, kWave - 1);
}

// The ordered part of a round, lane = slot.  A round is up to 64 slots, each a fragment of a pixel (lane `pixel` of the wave).  Only the
// carried state goes from slot to slot: a turn hands every slot the state behind the one in front of it in its pixel's order
// (slot_before; its own number: none of the round is), so after `turns` turns, as many as a pixel has slots at most, all have the right
// one; those that have it already make it again.  The rest of a fragment is worked out once, by its slot.
// last_slot: the last of the slots of the calling lane's own pixel, or -1.  Slots that are none have o = 0 and their own number.
// (Before, the lanes of the pixels walked their slots, and a step, of three or four a round, was 60 instructions that read a fragment's
// values from LDS and left the seed there; a turn is 24 now.  Saved order: 493 M vector instructions -> 460 M, 10^6 triangles 973 us ->
// 960, tile order 357 -> 349.)
template <bool kDepth, typename Take>
__device__ __forceinline__ ChainState taken(const ChainState &st, const Take &take) {
    ChainState t;
    t.alpha = take(st.alpha);
    t.s0 = take(st.s0); t.s1 = take(st.s1); t.s2 = take(st.s2);
    if constexpr (kDepth) { t.oa = take(st.oa); t.zoa = take(st.zoa); }
    return t;
}
template <bool kDepth>
__device__ __forceinline__ FragSeed walk_chain(const FragValue &v, int pixel, int slot_before, int turns, int last_slot, BackState &st) {
    const bool first = slot_before == (int)(threadIdx.x & (kWave - 1));
    const Remainder rem = remainder_of(v.o);
    const auto shared = [&](real x) { return __shfl(x, pixel, kWave); };
    ChainState in = taken<kDepth>(st, shared), out = chain_behind<kDepth>(in, v, rem.om, rem.inv);
    for (int turn = 1; turn < turns; turn++) {  // wave-uniform
        const ChainState handed = taken<kDepth>(out, [&](real x) { return __shfl(x, slot_before, kWave); });
        if (!first) in = handed;
        out = chain_behind<kDepth>(in, v, rem.om, rem.inv);
    }
    BackState of;  // the slot's pixel's
    of.g0 = shared(st.g0); of.g1 = shared(st.g1); of.g2 = shared(st.g2); of.g3 = shared(st.g3);
    of.final_alpha = shared(st.final_alpha);
    if constexpr (kDepth) {
        of.gd = shared(st.gd);
        of.final_weight = shared(st.final_weight); of.final_depth = shared(st.final_depth); of.inv_final_weight = shared(st.inv_final_weight);
    }
    const FragSeed f = fragment_seed<kDepth>(in, out, v, rem.inv, of);
    const int from = max(last_slot, 0);
    const ChainState end = taken<kDepth>(out, [&](real x) { return __shfl(x, from, kWave); });
    if (last_slot >= 0) static_cast<ChainState &>(st) = end;
    return f;
}
// The value of the lane before; lane 0's own.
__device__ __forceinline__ int lane_before(int x) { return __builtin_amdgcn_update_dpp(x, x, 0x138, 0xf, 0xf, false); }  // wave_shr:1

// Tile-order backward.  All pixels of a tile share the list order, so a wave walks its tile's list backwards, 64 entries at a
// time, by itself:
//   1. which entries cover which pixel: the lane's 64-bit mask the forward pass saved, asked for an entry block ahead (or the inside
//      tests again); the wave's ballot per entry is the transpose of the lanes' masks;
//   2. the ballots become slot numbers: entries from the far end, lanes in order inside an entry, so every
//      (pixel, entry) hit of the wave owns one slot, slots are grouped by entry, and a lane's own hits have increasing numbers in
//      the order it must visit them (reverse blend order);
//   then, in rounds of 64 slots:
//   3. lane = pixel: tells its slots whose they are, and which one is in front of them;
//   4. lane = slot: gathers the record of its fragment (the entry's triangle and vertex numbers are in LDS), the ordered part
//      (walk_chain), the 21 gradient terms into a term matrix, where three groups of 21 lanes add up the runs of equal entry and
//      issue one global floating-point atomic per run and term.
// Before, a workgroup of four waves staged every entry's record in LDS, between two barriers a block, each wave evaluated its
// fragments where their pixels were (three or four turns a round with a third of the lanes busy), and 36 KB of LDS held the CU to
// four of them.  Now a slot's record is gathered where the fragment is evaluated, by all lanes, entries that cover no pixel of the
// wave are not read at all, and the waves share nothing: a workgroup is one of them (workgroup_waves), five a SIMD.  us, both with
// dense gradient arrays: 10^6 triangles 603 -> 577, a mesh of 1.3 million 618 -> 440, 10^5 98 -> 82, 200 000 large ones 245 -> 224,
// 33 000 in tiles of 8 x 8 203 -> 87.  Asking for a block's vertex numbers a block ahead too leaves seven more registers in scratch
// memory (mesh 479); 32-bit byte offsets in the gather are ten operations less and change nothing.
struct TileWave {                // what a wave keeps in LDS
    real term[kTerms * kTermStride];
    alignas(16) int id[kBackBatch][4];  // the entries' triangles and vertices
    uint64_t ballot[kBackBatch]; // the lanes an entry covers
    uint32_t base[kBackBatch];   // an entry's first slot
    uint32_t tag[kWaveSlots];    // (entry | pixel's lane << 8 | slot in front of it in the pixel's order << 16) of a slot, its own where it is the first
};
template <int kLayout, bool kDepth, bool kPacked>
__global__ __launch_bounds__(kTileThreads, sizeof(real) != 4 ? 1 : kDepth ? 4 : 5) void backward_tile_order_kernel(RasterArgs a, BackwardArgs g) {
    extern __shared__ __align__(16) unsigned char s_dyn[];
    if (lists_invalid(g)) return;  // the same for the whole launch
    const int tid = threadIdx.x;
    int lane = tid & (kWave - 1);
    TileWave &mem = reinterpret_cast<TileWave *>(s_dyn)[tid / kWave];
    real *terms = mem.term;
    const TilePart group = part_of_workgroup();
    const TileId tile_id = tile_in_turn<kTileBandBackward, kEighths>(group.linear, gridDim.x, gridDim.y);
    const int slot_of_tile = group.part * blockDim.x + tid;
    const int tile = tile_id.index;
    const int start = a.offsets[tile];
    PixelCoord p = pixel_of_slot(a, tile_id.x, tile_id.y, slot_of_tile);
    p.ix = __builtin_amdgcn_readfirstlane(p.ix);  // of the wave's first pixel: all that wave_rect needs, and no register
    p.iy = __builtin_amdgcn_readfirstlane(p.iy);
    const TermLane tl = term_lane<kLayout>(g, lane);

    // With the forward pass's masks comes the number of list entries its workgroup has walked; else it is the largest `last` of my pixels.
    const bool saved_masks = g.hit_masks != nullptr;
    const int64_t mask_slots = (int64_t)g.mask_parts * g.mask_threads;
    const int first_slot = __builtin_amdgcn_readfirstlane(slot_of_tile);  // of the wave
    const uint64_t *const masks = g.hit_masks + (int64_t)gridDim.x * gridDim.y * g.mask_parts + first_slot;
    const int my_last = p.valid ? g.last[p.index] : 0;  // entries [0, my_last) of the list may hold my fragments
    BackState st = load_back_state<kDepth>(g, p.valid ? p.index : 0);  // of some pixel where there is none: slots that are none go through the walk as well
    int list_last = saved_masks ? (int)(int64_t)g.hit_masks[(int64_t)tile * g.mask_parts + first_slot / g.mask_threads] : -1;
    if (list_last < 0) list_last = wave_max_i32(my_last);  // no masks, or its pixels were rendered by several workgroups
    list_last = __builtin_amdgcn_readfirstlane(list_last);
    if (list_last == 0) return;

    // Blocks are aligned to multiples of kBackBatch from the start of the list (the last one may be short), so that a block is a whole
    // word of the saved hit masks.  What a block needs is asked for while the one before it is worked on.
    const int lo0 = (list_last - 1) / kBackBatch * kBackBatch;
    const auto triangle_at = [&](int lo) { return a.sorted_ids[start + min(max(lo, 0) + lane, list_last - 1)]; };
    const auto mask_at = [&](int lo) { return saved_masks && lo >= 0 && lo < my_last ? masks[hit_mask_chunk(start, tile, lo) * mask_slots + (uint32_t)lane] : 0ull; };
    const auto ids_of = [&](int tri) { const int32_t *v = a.indices + 3 * (int64_t)tri; return TriIds{tri, v[0], v[1], v[2]}; };
    uint64_t next_mask = mask_at(lo0);
    int next_triangle = triangle_at(lo0);
    for (int lo = lo0; lo >= 0; lo -= kBackBatch) {
        asm volatile("" : "+v"(lane));  // what depends on it is made here, not kept in registers by the loop
        const int nb = min(kBackBatch, list_last - lo);
        const int mine = my_last - lo;  // entries [0, mine) of this block are within my range
        const int triangle = next_triangle;
        uint64_t m = next_mask;
        next_triangle = triangle_at(lo - kBackBatch);
        next_mask = mask_at(lo - kBackBatch);
        if (__builtin_amdgcn_ballot_w64(mine > 0) != 0) {
            const TriIds ids = ids_of(triangle);
            // 1. which entries cover which pixel
            if (!saved_masks) {
                real t[9];
#pragma unroll
                for (int k = 0; k < 9; k++) t[k] = matrix_of<kPacked>(a, triangle)[k];
                uint64_t hit;
                PixelCoord q = p;
                asm volatile("" : "+v"(q.px), "+v"(q.py));  // the rectangle is made of them here: kept by the loop it is in scratch memory
                m = wave_hits(t, lane < nb, ((a.tw | a.th) & 7) == 0, wave_rect(a, q), q.px, q.py, hit, lane);
            }
            if (mine < kBackBatch) m &= mine > 0 ? (1ull << mine) - 1 : 0ull;  // entries past my last one
            // 2. slot numbers: lane = entry
            const uint64_t covered = transpose_bits(m, lane);
            const uint32_t count = (uint32_t)__builtin_popcountll(covered), incl = wave_inclusive_scan_u32(count);
            const uint32_t n_hits = (uint32_t)__builtin_amdgcn_readlane((int)incl, kWave - 1);
            mem.ballot[lane] = covered;
            mem.base[lane] = n_hits - incl;
            *reinterpret_cast<TriIds *>(mem.id[lane]) = ids;
            wave_lds_sync();

            for (uint32_t round0 = 0; round0 < n_hits; round0 += kWaveSlots) {
                const int n_slots = (int)min((uint32_t)kWaveSlots, n_hits - round0);
                // 3. whose the round's slots are
                int last_slot = -1, turns = 0;
                for (int handed_out = 0; handed_out < n_slots; turns++) {  // a turn hands out one at least: the first one left is its pixel's next
                    const int e = m ? top_bit(m) : 0;
                    const uint32_t slot = mem.base[e] + lanes_below_mask(mem.ballot[e]) - round0;
                    const bool there = m != 0 && slot < (uint32_t)kWaveSlots;
                    handed_out += __builtin_popcountll(__builtin_amdgcn_ballot_w64(there));
                    if (there) {
                        mem.tag[slot] = (uint32_t)e | (uint32_t)lane << 8 | (last_slot >= 0 ? (uint32_t)last_slot : slot) << 16;
                        last_slot = (int)slot;
                        m &= ~(1ull << e);
                    }
                }
                wave_lds_sync();

                // 4. the fragments' values, the ordered part, the terms
                const bool active = lane < n_slots;
                const uint32_t tag = active ? mem.tag[lane] : (uint32_t)lane << 8 | (uint32_t)lane << 16;
                const int entry = (int)(tag & 0xff), pixel = (int)(tag >> 8 & 0xff), slot_before = (int)(tag >> 16);
                const real px = __shfl(p.px, pixel, kWave), py = __shfl(p.py, pixel, kWave);
                BackRecord<kDepth> r;
                real b0 = 0.0f, b1 = 0.0f, b2 = 0.0f;
                FragValue value;
                value.o = value.color[0] = value.color[1] = value.color[2] = value.z = 0.0f;
                if (active) {
                    if constexpr (kPacked) gather_packed(a, mem.id[entry][0], r);
                    else gather_back(a, *reinterpret_cast<const TriIds *>(mem.id[entry]), r);
                    bary_apply(r.m, px, py, b0, b1, b2);
                    value = fragment_value(r, b0, b1, b2);
                }
                const FragSeed f = walk_chain<kDepth>(value, pixel, slot_before, turns, last_slot, st);
                if (active) {
                    real term[kTerms];
                    fragment_terms(f, r, b0, b1, b2, px, py, term);
#pragma unroll
                    for (int q = 0; q < kTerms; q++) terms[q * kTermStride + lane] = term[q];
                }
                const int entry_before = __shfl_up(entry, 1, kWave);
                const uint64_t heads = __builtin_amdgcn_ballot_w64(active && (lane == 0 || entry != entry_before));
                wave_lds_sync();
                add_run_sums(terms, n_slots, heads, tl, [&](int c, int v) { return mem.id[mem.tag[c] & 0xff][1 + v]; });
                wave_lds_sync();
            }
        }
    }
}

// list positions whose gradient sums are kept in LDS by the per-pixel-order kernel (the double build has
// half the room per scalar and twice the candidate lists)
constexpr int kAccWindow = sizeof(real) == 4 ? 512 : 128;

// The order the reverse selection walks: by pixel depth, a NaN depth behind every number (that is where the
// forward selection leaves such a fragment, render.cu:338-373: every comparison with it is false), equal
// depths (two NaNs count as equal) by list position.
__device__ __forceinline__ bool depth_before(real a, real b) { return a < b || (b != b && a == a); }
__device__ __forceinline__ bool depth_same(real a, real b) { return a == b || (a != a && b != b); }

// Candidate insertion for the reverse selection: keeps the `cap` LARGEST
// (depth, position) pairs in descending order.  Positions arrive in ascending
// order, so a candidate whose depth equals a stored one has the larger position
// and goes in front of it.
__device__ __forceinline__ void topk_insert_desc(const TopK &tk, int cap, int &n, real d, int j) {
    if (n == cap && depth_before(d, tk.d(cap - 1))) return;
    int i = (n < cap) ? n : cap - 1;
    while (i > 0 && !depth_before(d, tk.d(i - 1))) {
        tk.d(i) = tk.d(i - 1);
        tk.j(i) = tk.j(i - 1);
        i--;
    }
    tk.d(i) = d;
    tk.j(i) = j;
    if (n < cap) n++;
}

template <int kLayout>
__global__ __launch_bounds__(kTileThreads) void backward_pixel_order_kernel(RasterArgs a, BackwardArgs g) {
    extern __shared__ __align__(16) unsigned char s_dyn[];
    const int n_threads = blockDim.x;
    DepthRecord *s_rec = reinterpret_cast<DepthRecord *>(s_dyn);
    TopK tk;
    tk.depth = reinterpret_cast<real *>(s_dyn + sizeof(DepthRecord) * kBatch);
    tk.pos = reinterpret_cast<int *>(tk.depth + kLayers * n_threads);
    tk.n_threads = n_threads;
    // Per-entry sums of the first kAccWindow list positions live in LDS and are
    // flushed once per tile; positions beyond the window go straight to memory.
    real *s_acc = reinterpret_cast<real *>(tk.pos + kLayers * n_threads);

    __shared__ uint8_t s_touch[kBatch];
    __shared__ WaveRect s_rects[kMaxTileWaves];
    if (lists_invalid(g)) return;  // the same for the whole launch
    const int tid = threadIdx.x;
    const int wave = tid / kWave;
    const int n_waves = blockDim.x / kWave;
    const TileId tile_id = tile_of_workgroup<kTileBandBackward, kEighths>();
    const int tile = tile_id.index;
    const int start = a.offsets[tile], end = a.offsets[tile + 1];
    const PixelCoord p = pixel_of_thread(a, tile_id);
    publish_wave_rect(a, p, s_rects);
    const bool tests_small = tests_small_entries(a, end - start, (int)(gridDim.x * gridDim.y));
    const int n_acc = min(end - start, kAccWindow);
    for (int i = tid; i < n_acc * kTerms; i += blockDim.x) s_acc[i] = 0.0f;

    BackState st;
    int remaining = 0;
    // exclusive upper bound of the fragments still to visit, in (depth, position) order
    real bound_depth = 0.0f;
    int bound_j = 0;
    if (p.valid) {
        st = load_back_state<true>(g, p.index);
        remaining = min(g.ends[p.index], a.max_layers);  // render.cu:642
        bound_depth = g.last_depth[p.index];
        bound_j = start + g.last[p.index];  // one past the last blended entry
    }
    while (true) {
        const bool want = remaining > 0;
        if (!__syncthreads_or(want)) break;
        const int cap = min(kLayers, remaining);
        int found = 0;
        for (int batch = start; batch < end; batch += kBatch) {
            const int nb = min(kBatch, end - batch);
            __syncthreads();
            for (int e = tid; e < nb; e += blockDim.x) {
                gather_depth<false>(a, batch + e, s_rec[e]);
                s_touch[e] = (uint8_t)(waves_touched(s_rec[e].m, s_rects, n_waves) | small_entry(a, s_rec[e].extent, tests_small));
            }
            __syncthreads();
            uint64_t m[kBatch / kWave];
            batch_hit_mask<kBatch / kWave>(s_rec, s_touch, s_rects, nb, wave, p.px, p.py, m);
            if (!want) {
#pragma unroll
                for (int wd = 0; wd < kBatch / kWave; wd++) m[wd] = 0;
            }
            while (true) {
                const int e = pop_lowest<kBatch / kWave>(m);
                if (__builtin_amdgcn_ballot_w64(e >= 0) == 0) break;  // wave-uniform
                if (e < 0) continue;
                const DepthRecord &r = s_rec[e];
                real b0, b1, b2;
                bary_apply(r.m, p.px, p.py, b0, b1, b2);
                const real pd = interp_w(b0, b1, b2, r.z[0], r.z[1], r.z[2], r.w[0], r.w[1], r.w[2]);
                const int j = batch + e;
                if (depth_before(pd, bound_depth) || (depth_same(pd, bound_depth) && j < bound_j)) topk_insert_desc(tk, cap, found, pd, j);
            }
        }
        if (want) {
            for (int i = 0; i < found; i++) {
                BackRecord<true> r;
                gather_back(a, load_ids(a, tk.j(i)), r);
                real b0, b1, b2;
                bary_apply(r.m, p.px, p.py, b0, b1, b2);
                if (!bary_inside(b0, b1, b2)) continue;  // cannot happen: the selection tested it
                real term[kTerms];
                fragment_backward(st, r, b0, b1, b2, p.px, p.py, term);
                const int rel = tk.j(i) - start;
                if (rel < kAccWindow) {
#pragma unroll
                    for (int q = 0; q < kTerms; q++) atomicAdd(s_acc + rel * kTerms + q, term[q]);
                } else {
#pragma unroll
                    for (int q = 0; q < kTerms; q++)
                        if (term[q] != 0.0f) unsafeAtomicAdd(term_address<kLayout>(g, r.id[q / 7], q % 7), term[q]);
                }
            }
            if (found < cap) {
                remaining = 0;  // list exhausted
            } else {
                remaining -= found;
                bound_depth = tk.d(found - 1);
                bound_j = tk.j(found - 1);
            }
        }
    }
    __syncthreads();
    for (int e = tid; e < n_acc; e += blockDim.x) {
        const TriIds t = load_ids(a, start + e);
        const int id[3] = {t.ia, t.ib, t.ic};
#pragma unroll
        for (int q = 0; q < kTerms; q++) {
            const real v = s_acc[e * kTerms + q];
            if (v != 0.0f) unsafeAtomicAdd(term_address<kLayout>(g, id[q / 7], q % 7), v);
        }
    }
}

// Per-pixel order with the blend order saved by the forward pass
// (max_layers <= TG_MAX_SAVED_LAYERS): no re-selection.  Step s of a pixel is its
// fragment n - 1 - s, so every pixel starts at its own far end.  The pixels of a wave
// hold different numbers of fragments, so the wave takes its (pixel, step) pairs 64 at a
// time: a round's 64 slots keep every lane busy whatever the pixels' counts are.  A round
// takes the pending pairs nearest the far end of the tile's list (every pixel a prefix of
// its next steps): the slots of a round then hold few different entries.  Per round:
//   1. lane = pixel: which of my next steps (their list positions are fetched from the
//      saved order kPrefix steps ahead) lie at or above the round's threshold; they get
//      consecutive slots;
//   2. lane = slot: the slots are grouped by entry (ballot matching); a slot takes the
//      lane, and the column of the term matrix, that this gives it;
//   3. lane = column: gathers the record of its fragment from memory (neighbouring
//      pixels hold the same few entries, so the loads hit in cache; staging the tile's
//      records in LDS first was measured slower, for the workgroups per CU it costs);
//   4. the ordered part (walk_chain);
//   5. the 21 gradient terms into the term matrix, where three groups of 21 lanes add up
//      the runs of equal entry and issue one global floating-point atomic per run and term
//      (LDS floating-point atomics cost about three cycles per lane on gfx950).
// Grouped before the gather and not behind it, four neighbouring lanes, whose addresses the CU takes together, mostly ask for the
// same lines: 27 lines a load and atomic -> 18, the address unit busy 70 % of the time -> 63.  With the walk by slots (walk_chain), us:
// 10^6 triangles 958 -> 930, 20 000 without a limit on the layers 523 -> 500, 200 000 large ones 218 -> 210, 33 000 in tiles of 8 x 8
// 114 -> 110.
// The waves of a tile share nothing, so a workgroup is one of them: its place is free for another tile's when it is done, where
// workgroups of four wait for the longest of them (workgroup_waves).  In fours and so, us: 10^6 triangles 1057, 1013, 10^5 83.5, 76,
// 20 000 with a heavy tail on 1920 x 1080 61, 55, a mesh of 1.3 million 185, 180.
// What a wave keeps in LDS.  A workgroup takes it for the waves it has (taken for four always, frames in tiles of 8 x 8, a wave each,
// had five workgroups a CU: 33 000 triangles 229 us, so 116).
// Steps that a pixel can have in a round.  Fewer are fewer turns of the walk and candidates for a slot, and rounds of more entries (us, 4, 3,
// 2 steps: 10^6 triangles 942, 912, 947, 20 000 without a limit on the layers 498, 470, 465, a mesh of 1.3 million 175, 177, 184, 10^5 73, 73, 80).
// With 3, asked for where they stay (fetch_behind) and the pixel's own values after them: 896, 470, 177, 73; 33 000 in tiles of 8 x 8 109 -> 105.
constexpr int kPrefix = 3;
constexpr int kNotFirst = 0x80;  // the slot before is one of the same pixel
struct SavedWave {
    real term[kTerms * kTermStride];
    int rel[kWave];         // list position of a slot's fragment, from the tile's start
    int vertex[3 * kWave];  // the three vertex ids of a column's entry
    uint8_t src[kWave];     // the pixel (lane) of a slot, and kNotFirst
};
template <int kLayout, bool kDepth, bool kPacked>
__global__ __launch_bounds__(kTileThreads, sizeof(real) != 4 ? 1 : kDepth || kLayout == kGradStrided ? 4 : 5) void backward_saved_order_kernel(RasterArgs a, BackwardArgs g) {
    extern __shared__ __align__(16) unsigned char s_dyn[];
    if (lists_invalid(g)) return;  // the same for the whole launch
    const int tid = threadIdx.x;
    int lane = tid & (kWave - 1);
    SavedWave &mem = reinterpret_cast<SavedWave *>(s_dyn)[tid / kWave];
    const TilePart group = part_of_workgroup();
    const TileId tile_id = g.deep ? tile_in_turn<kTileBandBackward, kSixteenths>(group.linear, gridDim.x, gridDim.y)
                                  : tile_in_turn<kTileBandBackward, kEighths>(group.linear, gridDim.x, gridDim.y);
    const int slot_of_tile = group.part * blockDim.x + tid;
    const int tile = tile_id.index;
    const int start = a.offsets[tile], end = a.offsets[tile + 1];
    const PixelCoord p = pixel_of_slot(a, tile_id.x, tile_id.y, slot_of_tile);
    const int rel_bits = 32 - __builtin_clz(max(end - start - 1, 1));  // bits that tell two list positions apart
    real *terms = mem.term;
    int *vertices = mem.vertex;
    const TermLane tl = term_lane<kLayout>(g, lane);

    int n = 0;
    if (p.valid) {
        // render.cu:642; fewer than were blended only where a NaN depth had the list blended more than once
        n = min(g.ends[p.index], min(a.max_layers, order_rows(g.order, a, end - start)));
    }
    const int64_t plane = order_stride(g.order, a);
    const bool long_list = end - start > kShortList;  // then the positions' high halves were saved as well
    // The list positions of my next three steps, -1 where there is none: below every threshold.  Step s is layer n - 1 - s, so the next
    // one is `next_layer`, the others lie a plane further down each.
    const uint16_t *next_layer = g.order.low + ((int64_t)(n - 1) * plane + order_first(g.order, p, start, slot_of_tile));
    const int64_t high_halves = g.order.high;
    int steps_left = n;
    int ahead[kPrefix];
    // The first `kept` of them are there; the others are asked for.  (Each into the register it stays in: one that is moved is waited for,
    // and while every step taken moved all of them a round waited for as many loads, one after the other, as a pixel had steps in it.)
    auto fetch_behind = [&](int kept) {
#pragma unroll
        for (int i = 0; i < kPrefix; i++)
            if (kept <= i) {
                ahead[i] = -1;
                if (i < steps_left) {
                    const uint16_t *layer = next_layer - i * plane;
                    ahead[i] = *layer;
                    if (long_list) ahead[i] |= (int)layer[high_halves] << 16;
                }
            }
    };
    fetch_behind(0);
    BackState st = load_back_state<kDepth>(g, p.valid ? p.index : 0);  // of some pixel where there is none: slots that are none go through the walk as well
    int remaining = __builtin_amdgcn_readlane((int)wave_inclusive_scan_u32((uint32_t)n), kWave - 1);  // the wave's fragments not handed out yet

    // How many of my next steps lie at or above list position `threshold`: a prefix of them, so that I visit them in order.
    // -> the slots that makes.
    auto slots_at = [&](int threshold) {
        uint64_t lanes = ~0ull;
        int slots = 0;
#pragma unroll
        for (int i = 0; i < kPrefix; i++) {
            lanes &= __builtin_amdgcn_ballot_w64(ahead[i] >= threshold);
            slots += __builtin_popcountll(lanes);
        }
        return slots;
    };

    int span = end - start;  // list positions of the last round, from its threshold to its largest
    for (int round = 0; remaining > 0; round++) {
        asm volatile("" : "+v"(lane));  // what depends on it is made here, not kept in registers by the loop
        // 1. the round's slots.  A round takes the wave's pending fragments from the far end of the tile's LIST, not step s
        //    of every pixel: a triangle is at another step in each pixel it covers, but at one list position, so the
        //    slots of a round then hold few different entries -- long runs, few atomics, and gathers whose lanes share
        //    their cache lines.  Every pixel gives a prefix of its next (at most kPrefix) steps, those at or above a
        //    threshold: the largest threshold that fills the 64 slots.  What overflows is cut off in lane order from a
        //    start lane that moves from round to round, and waits for the next round.
        int threshold = 0, offered = slots_at(0), match_bits = rel_bits;
        if (offered > kWave) {
            const int top = wave_max_i32(ahead[0]) + 1;
            int high = top;  // slots_at(threshold) >= 64 > slots_at(high) = 0
            int middle = high - 2 * span;  // first twice what the last round took, then halves
            while (high - threshold > 1) {
                if (middle <= threshold) middle = threshold + (high - threshold) / 2;
                const int slots = slots_at(middle);
                if (slots >= kWave) { threshold = middle; offered = slots; } else { high = middle; }
                middle = 0;
            }
            span = max(top - threshold, 1);
            match_bits = 32 - __builtin_clz(span);
        }
        int mine_count = 0;
#pragma unroll
        for (int i = 0; i < kPrefix; i++) mine_count += mine_count == i && ahead[i] >= threshold;
        const int taken_incl = (int)wave_inclusive_scan_u32((uint32_t)mine_count);
        const int first_lane = (round * 23) & (kWave - 1);
        const int before_first = __builtin_amdgcn_readlane(taken_incl - mine_count, first_lane);
        int base = taken_incl - mine_count - before_first;
        if (lane < first_lane) base += offered;
        const int granted = max(0, min(mine_count, kWave - base));
        const int n_slots = min(kWave, offered);
        int *rels = mem.rel;
        uint8_t *srcs = mem.src;
        // my slots of the round: neighbours, increasing slot = increasing step
        int turns = 1;
#pragma unroll
        for (int i = 0; i < kPrefix; i++) {
            if (granted > i) { rels[base + i] = ahead[i]; srcs[base + i] = (uint8_t)(i ? lane | kNotFirst : lane); }
            if (i) turns += __builtin_amdgcn_ballot_w64(granted > i) != 0;
        }
        const int last_slot = granted > 0 ? base + granted - 1 : -1;
#pragma unroll
        for (int i = 0; i + 1 < kPrefix; i++)
#pragma unroll
            for (int k = 1; i + k < kPrefix; k++)
                if (granted == k) ahead[i] = ahead[i + k];
        steps_left -= granted;
        next_layer -= granted * plane;
        if (granted > 0) fetch_behind(kPrefix - granted);
        remaining -= n_slots;
        wave_lds_sync();

        // 2. The slots grouped by entry (ballot matching, groups in the order of their lowest slot): the column a slot takes.
        const bool active = lane < n_slots;
        const int src = active ? srcs[lane] : lane;
        int rel = active ? rels[lane] : 0;
        // By the bits that tell positions of the round's range apart: the few positions outside it (a second step behind a
        // first one, by depth, may come later in the list) can be taken together with others, and then make more runs, not
        // other ones.
        uint64_t peers = __builtin_amdgcn_ballot_w64(active);
        for (int b = 0; b < match_bits; b++) {  // wave-uniform
            const int bit = bit_mask(rel, b);
            const uint64_t vote = __builtin_amdgcn_ballot_w64(bit != 0);
            peers &= ~(vote ^ (uint64_t)(int64_t)bit);
        }
        const uint32_t rank = lanes_below_mask(peers);
        const uint32_t size = active && rank == 0 ? (uint32_t)__builtin_popcountll(peers) : 0u;
        const uint32_t incl = wave_inclusive_scan_u32(size);
        int column = __shfl((int)(incl - size), active ? __builtin_ctzll(peers) : lane, kWave) + (int)rank;
        if (!active) column = lane;
        const int last_column = __shfl(column, max(last_slot, 0), kWave);
        const int before = lane_before(column);
        int tag = (src & (kWave - 1)) | ((src & kNotFirst) ? before : column) << 8;
        tag = __builtin_amdgcn_ds_permute(column * 4, tag);
        rel = __builtin_amdgcn_ds_permute(column * 4, rel);
        const int pixel = tag & 0xff, slot_before = tag >> 8;

        // 3. lane = column: the record, and the fragment's own values
        const real px = __shfl(p.px, pixel, kWave), py = __shfl(p.py, pixel, kWave);
        BackRecord<kDepth> r;
        real b0 = 0.0f, b1 = 0.0f, b2 = 0.0f;
        FragValue value;
        value.o = value.color[0] = value.color[1] = value.color[2] = value.z = 0.0f;
        if (active) {
            if constexpr (kPacked) gather_packed(a, a.sorted_ids[start + rel], r);
            else gather_back(a, load_ids(a, start + rel), r);
            bary_apply(r.m, px, py, b0, b1, b2);
            value = fragment_value(r, b0, b1, b2);
        }
        // 4. the ordered part
        const FragSeed f = walk_chain<kDepth>(value, pixel, slot_before, turns, last_slot >= 0 ? last_column : -1, st);
        // 5. the terms
        if (active) {
            real term[kTerms];
            fragment_terms(f, r, b0, b1, b2, px, py, term);
#pragma unroll
            for (int q = 0; q < kTerms; q++) terms[q * kTermStride + lane] = term[q];
#pragma unroll
            for (int k = 0; k < 3; k++) vertices[k * kWave + lane] = r.id[k];
        }
        // a column starts a run where its entry differs from the column before
        const int rel_before = lane_before(rel);
        const uint64_t heads = __builtin_amdgcn_ballot_w64(active && (lane == 0 || rel != rel_before));
        wave_lds_sync();
        add_run_sums(terms, n_slots, heads, tl, [&](int c, int v) { return vertices[v * kWave + c]; });
        wave_lds_sync();
    }
}

// The instances that read triangles' records, of frames in one call: gradients dense or in (V,8) blocks.  Null in the double build, which
// has no such frames.
using BackwardKernel = void (*)(RasterArgs, BackwardArgs);
BackwardKernel packed_tile_order_backward(GradLayout layout, bool depth);
BackwardKernel packed_saved_order_backward(GradLayout layout, bool depth);

}  // namespace tg
