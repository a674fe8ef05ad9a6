// tg_gradient_copies.hpp -- the (V,8) blocks that a frame's gradients are summed in: the library's rule, and the torch module's, which
// allocates them.  Why the lines lie where they do is said where the blocks are used (tg_frame_backward).
// Of the keys that were counted, not of the ones there is room for: a key buffer has room for an eighth and 1024 more, a first frame's for
// 65536 more, and a plan serves later frames with a fraction of its keys.
#pragma once
#include "../../include/trigrad_hip.h"

namespace tg {

inline int gradient_copies(const tg_frame &f) {
    const int64_t pixels = f.width * f.height, waves_of_a_tile = (f.tile_w * f.tile_h + 63) / 64;
    const bool shared = 3 * f.n_triangles > 2 * f.n_vertices;  // vertices are several triangles'
    const bool by_xcd = !f.per_pixel_sort || (f.flags & (TG_FRAME_ORDER_PLANES | TG_FRAME_ORDER_POOL));  // without a saved order the kernel knows one block
    if (by_xcd && pixels > 16384 && pixels >= 4 * f.n_vertices && f.n_vertices <= 131072 && f.n_keys * waves_of_a_tile >= 20 * f.n_triangles) return 8;
    if (f.per_pixel_sort) return pixels > 16384 || f.n_vertices >= 32768;
    return (shared && pixels > 65536) || (f.n_vertices >= 32768 && pixels >= 1 << 19);
}

}  // namespace tg
