// tg_camera.hip -- the step in front of the renderer: near-plane splitting and the division by w.
//
// Both are bound by memory traffic, and by how often it is paid: as tensor operations the splitting of 200 000
// triangles (half of them behind the plane) was 230 launches and nine host reads, 1500 us, for 18 MB in and out.
// Here it is two launches with one host read between them, because the number of output triangles decides the size
// of the output arrays:
//   clip_count_kernel   per workgroup of kClipTile triangles, how many triangles leave it
//   clip_emit_kernel    the same triangles again: a workgroup adds up the totals of those before it, scans its own
//                       counts, and every thread writes the triangles of its own (at most two each)
// The arithmetic is that of the tensor operations, one rounding per operation in the same order.
#include "tg_raster.hpp"

namespace tg {

constexpr int kClipThreads = 256;
constexpr int kClipRounds = 4;                            // triangles per thread
constexpr int kClipTile = kClipThreads * kClipRounds;
constexpr uint32_t kClipBadIndex = 0x80000000u;           // in a workgroup's total: it saw an index outside the vertices

// Signed distances of a triangle's corners to the plane z + w = 0 and which of them are kept.
struct ClipTriangle {
    int id[3];
    real d[3];
    uint32_t inside;  // bit k: corner k
    bool ok;
};

__device__ __forceinline__ ClipTriangle clip_triangle(const real4 *__restrict__ clip, int n_vertices, const int32_t *__restrict__ indices,
                                                      int64_t t) {
    ClipTriangle r;
    r.inside = 0;
    r.ok = true;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        int i = indices[3 * t + k];
        if (i < 0) i += n_vertices;  // as a tensor index counts
        const bool ok = (unsigned)i < (unsigned)n_vertices;
        r.ok = r.ok && ok;
        r.id[k] = ok ? i : 0;
    }
    if (!r.ok) return r;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const real4 v = clip[r.id[k]];
        r.d[k] = v.z + v.w;
        if (r.d[k] >= 0.0f) r.inside |= 1u << k;
    }
    return r;
}

// Triangles that come out of one: none, itself, one cut off at a corner, or the two of a quadrangle.
__device__ __forceinline__ uint32_t clip_pieces(uint32_t inside) {
    const int kept = __builtin_popcount(inside);
    return kept == 0 ? 0u : kept == 2 ? 2u : 1u;
}

__global__ __launch_bounds__(kClipThreads) void clip_count_kernel(const real4 *__restrict__ clip, int n_vertices,
                                                                  const int32_t *__restrict__ indices, int64_t n_triangles,
                                                                  uint32_t *__restrict__ totals, uint32_t *__restrict__ host_totals) {
    __shared__ uint32_t s_wave[kClipThreads / kWave];
    uint32_t count = 0;
    bool bad = false;
#pragma unroll
    for (int k = 0; k < kClipRounds; k++) {
        const int64_t t = (int64_t)blockIdx.x * kClipTile + k * kClipThreads + threadIdx.x;
        if (t < n_triangles) {
            const ClipTriangle c = clip_triangle(clip, n_vertices, indices, t);
            bad = bad || !c.ok;
            count += clip_pieces(c.inside);
        }
    }
    const uint32_t incl = wave_inclusive_scan_u32(count);
    const bool wave_bad = __builtin_amdgcn_ballot_w64(bad) != 0;
    if ((threadIdx.x & (kWave - 1)) == kWave - 1) s_wave[threadIdx.x / kWave] = incl | (wave_bad ? kClipBadIndex : 0u);
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t sum = 0, flags = 0;
        for (int w = 0; w < kClipThreads / kWave; w++) {
            sum += s_wave[w] & ~kClipBadIndex;
            flags |= s_wave[w] & kClipBadIndex;
        }
        totals[blockIdx.x] = sum;
        host_totals[blockIdx.x] = sum | flags;
    }
}

struct ClipOut {
    real4 *vertices;
    int32_t *indices;
    real *colors;
    real *opacities;
};

// One output vertex: corner `from` of the triangle, or (cut) the point where its edge to corner `to` meets the plane.
template <int kColors, int kOpacities>  // scalars per vertex; 0: the run-time width
__device__ __forceinline__ void clip_vertex(const real4 *__restrict__ clip, const real *__restrict__ colors, int color_width,
                                            const real *__restrict__ opacities, int opacity_width, const ClipOut &out, int64_t at,
                                            bool cut, int from, int to, real d_from, real d_to) {
    const int nc = kColors ? kColors : color_width, no = kOpacities ? kOpacities : opacity_width;
    const real t = d_from / (d_from - d_to);
    real4 v = clip[from];
    if (cut) {
        const real4 b = clip[to];
        v = make_real4(v.x + t * (b.x - v.x), v.y + t * (b.y - v.y), v.z + t * (b.z - v.z), v.w + t * (b.w - v.w));
    }
    out.vertices[at] = v;
    for (int k = 0; k < nc; k++) {
        real x = colors[(int64_t)from * nc + k];
        if (cut) x = x + t * (colors[(int64_t)to * nc + k] - x);
        out.colors[at * nc + k] = x;
    }
    for (int k = 0; k < no; k++) {
        real x = opacities[(int64_t)from * no + k];
        if (cut) x = x + t * (opacities[(int64_t)to * no + k] - x);
        out.opacities[at * no + k] = x;
    }
}

__device__ __forceinline__ int pick3(int k, int a, int b, int c) { return k == 0 ? a : k == 1 ? b : c; }
__device__ __forceinline__ real pick3(int k, real a, real b, real c) { return k == 0 ? a : k == 1 ? b : c; }

template <int kColors, int kOpacities>
__global__ __launch_bounds__(kClipThreads) void clip_emit_kernel(const real4 *__restrict__ clip, int n_vertices,
                                                                 const int32_t *__restrict__ indices, int64_t n_triangles,
                                                                 const real *__restrict__ colors, int color_width,
                                                                 const real *__restrict__ opacities, int opacity_width,
                                                                 const uint32_t *__restrict__ totals, int64_t n_out, ClipOut out) {
    __shared__ uint32_t s_before[kClipThreads / kWave], s_wave[kClipRounds][kClipThreads / kWave];
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    uint32_t before = 0;
    for (int b = tid; b < (int)blockIdx.x; b += kClipThreads) before += totals[b];
    before = wave_inclusive_scan_u32(before);
    if (lane == kWave - 1) s_before[wave] = before;
    ClipTriangle c[kClipRounds];
    uint32_t pieces[kClipRounds], incl[kClipRounds];
#pragma unroll
    for (int k = 0; k < kClipRounds; k++) {
        const int64_t t = (int64_t)blockIdx.x * kClipTile + k * kClipThreads + tid;
        c[k].inside = 0;
        if (t < n_triangles) c[k] = clip_triangle(clip, n_vertices, indices, t);
        pieces[k] = clip_pieces(c[k].inside);
        incl[k] = wave_inclusive_scan_u32(pieces[k]);
        if (lane == kWave - 1) s_wave[k][wave] = incl[k];
    }
    __syncthreads();
    int64_t base = 0;
#pragma unroll
    for (int w = 0; w < kClipThreads / kWave; w++) base += s_before[w];
#pragma unroll
    for (int k = 0; k < kClipRounds; k++) {
        int64_t at = base + incl[k] - pieces[k];
#pragma unroll
        for (int w = 0; w < kClipThreads / kWave; w++) {
            if (w < wave) at += s_wave[k][w];
            base += s_wave[k][w];
        }
        if (pieces[k] == 0 || at + pieces[k] > n_out) continue;
        const uint32_t inside = c[k].inside;
        const int kept = __builtin_popcount(inside);
        // corner s: the first one; with one corner kept the kept one, with two the one cut away.  r, q follow it.
        const int s = kept == 3 ? 0 : __builtin_ctz(kept == 1 ? inside : ~inside & 7u);
        const int q = s == 0 ? 1 : s == 1 ? 2 : 0, r = s == 0 ? 2 : s == 1 ? 0 : 1;
        const int is = pick3(s, c[k].id[0], c[k].id[1], c[k].id[2]), iq = pick3(q, c[k].id[0], c[k].id[1], c[k].id[2]),
                  ir = pick3(r, c[k].id[0], c[k].id[1], c[k].id[2]);
        const real ds = pick3(s, c[k].d[0], c[k].d[1], c[k].d[2]), dq = pick3(q, c[k].d[0], c[k].d[1], c[k].d[2]),
                   dr = pick3(r, c[k].d[0], c[k].d[1], c[k].d[2]);
#define TG_CLIP_VERTEX(corner, cut, from, to, d_from, d_to)                                                                       \
    clip_vertex<kColors, kOpacities>(clip, colors, color_width, opacities, opacity_width, out, 3 * at + (corner), cut, from, to, \
                                     d_from, d_to)
        if (kept != 2) {
            TG_CLIP_VERTEX(0, false, is, is, ds, ds);
            TG_CLIP_VERTEX(1, kept == 1, kept == 1 ? is : iq, iq, ds, dq);
            TG_CLIP_VERTEX(2, kept == 1, kept == 1 ? is : ir, ir, ds, dr);
        } else {
            TG_CLIP_VERTEX(0, false, iq, iq, dq, dq);
            TG_CLIP_VERTEX(1, false, ir, ir, dr, dr);
            TG_CLIP_VERTEX(2, true, iq, is, dq, ds);
            TG_CLIP_VERTEX(3, true, iq, is, dq, ds);
            TG_CLIP_VERTEX(4, false, ir, ir, dr, dr);
            TG_CLIP_VERTEX(5, true, ir, is, dr, ds);
        }
#undef TG_CLIP_VERTEX
        for (int i = 0; i < 3 * (int)pieces[k]; i++) out.indices[3 * at + i] = (int32_t)(3 * at + i);
    }
}

// (x, y, z, w) -> (x/w, y/w, z/w, 1/w), 32 bytes a vertex.
__global__ __launch_bounds__(kClipThreads) void clip_to_render_kernel(const real4 *__restrict__ clip, int64_t n, real4 *__restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * kClipThreads + threadIdx.x;
    if (i >= n) return;
    const real4 v = clip[i];
    out[i] = make_real4(v.x / v.w, v.y / v.w, v.z / v.w, (real)1.0 / v.w);
}

static int check_clip(const char *fn, const void *clip, int32_t n_vertices, const void *indices, int64_t n_triangles) {
    if (n_vertices < 0 || n_triangles < 0 || n_triangles > 0x7fffffffll * 256 || (n_triangles > 0 && (!clip || !indices)) ||
        ((uintptr_t)clip & 15)) {
        set_error("%s: null pointer, count out of range or clip coordinates not aligned to a row", fn);
        return TG_E_ARG;
    }
    return 0;
}

}  // namespace tg

using namespace tg;

extern "C" int64_t tg_clip_blocks(int64_t n_triangles) { return n_triangles < 0 ? 0 : ceil_div64(n_triangles, kClipTile); }

extern "C" int tg_clip_count(const real *clip, int32_t n_vertices, const int32_t *indices, int64_t n_triangles, uint32_t *totals,
                             uint32_t *host_totals, void *stream) {
    if (int e = check_clip("tg_clip_count", clip, n_vertices, indices, n_triangles)) return e;
    if (n_triangles == 0) return 0;
    if (!totals || !host_totals) { set_error("tg_clip_count: totals is null"); return TG_E_ARG; }
    TG_LAUNCH(clip_count_kernel, dim3((unsigned)tg_clip_blocks(n_triangles)), dim3(kClipThreads), 0, (hipStream_t)stream,
              (const real4 *)clip, n_vertices, indices, n_triangles, totals, host_totals);
    return check_launch("clip_count_kernel");
}

extern "C" int tg_clip_emit(const real *clip, int32_t n_vertices, const int32_t *indices, int64_t n_triangles, const real *colors,
                            int32_t color_width, const real *opacities, int32_t opacity_width, const uint32_t *totals, int64_t n_out,
                            real *out_clip, int32_t *out_indices, real *out_colors, real *out_opacities, void *stream) {
    if (int e = check_clip("tg_clip_emit", clip, n_vertices, indices, n_triangles)) return e;
    if (n_triangles == 0 || n_out == 0) return 0;
    if (n_out < 0 || n_out > 0x7fffffffll / 3 || color_width < 0 || opacity_width < 0 || !totals || !out_clip || !out_indices ||
        (color_width > 0 && (!colors || !out_colors)) || (opacity_width > 0 && (!opacities || !out_opacities)) ||
        ((uintptr_t)out_clip & 15)) {
        set_error("tg_clip_emit: null pointer, count out of range or misaligned output");
        return TG_E_ARG;
    }
    const ClipOut out{(real4 *)out_clip, out_indices, out_colors, out_opacities};
    const dim3 grid((unsigned)tg_clip_blocks(n_triangles));
    // the renderer's own widths (three colour channels, one opacity) address with constants
    if (color_width == 3 && opacity_width == 1)
        TG_LAUNCH_AS("clip_emit_kernel", (clip_emit_kernel<3, 1>), grid, dim3(kClipThreads), 0, (hipStream_t)stream, (const real4 *)clip,
                     n_vertices, indices, n_triangles, colors, color_width, opacities, opacity_width, totals, n_out, out);
    else
        TG_LAUNCH_AS("clip_emit_kernel", (clip_emit_kernel<0, 0>), grid, dim3(kClipThreads), 0, (hipStream_t)stream, (const real4 *)clip,
                     n_vertices, indices, n_triangles, colors, color_width, opacities, opacity_width, totals, n_out, out);
    return check_launch("clip_emit_kernel");
}

extern "C" int tg_clip_to_render(const real *clip, int64_t n_vertices, real *out, void *stream) {
    if (n_vertices < 0 || n_vertices > 0x7fffffffll * kClipThreads || (n_vertices > 0 && (!clip || !out)) || ((uintptr_t)clip & 15) ||
        ((uintptr_t)out & 15)) {
        set_error("tg_clip_to_render: null or misaligned pointer, or count out of range");
        return TG_E_ARG;
    }
    if (n_vertices == 0) return 0;
    TG_LAUNCH(clip_to_render_kernel, dim3((unsigned)ceil_div64(n_vertices, kClipThreads)), dim3(kClipThreads), 0, (hipStream_t)stream,
              (const real4 *)clip, n_vertices, (real4 *)out);
    return check_launch("clip_to_render_kernel");
}
