// Launch arguments of the frame products (yas_frame_dev.hpp).
#pragma once

#include "yas_frame_dev.hpp"

namespace yas {

// Levels base .. base + 2 (as far as there are any): from `base` > 0 on, the
// first of them is there already and is only read.  The caller sets a.src.
template <class Src>
inline void fill_image(ImageArgs<Src>& a, const Level* lv, int levels, int base, float* const* out, float* const* gx,
                       float* const* gy) {
  a.n = levels - base < kImageLevels ? levels - base : kImageLevels;
  for (int i = 0; i < kImageLevels; ++i) {
    const int l = base + (i < a.n ? i : 0);
    a.w[i] = lv[l].w;
    a.h[i] = lv[l].h;
    a.out[i] = i < a.n && (i > 0 || base == 0) ? out[l] : nullptr;
    a.gx[i] = gx ? gx[l] : nullptr;
    a.gy[i] = gy ? gy[l] : nullptr;
  }
  a.tiles_x = (a.w[0] + kImageTile - 1) / kImageTile;
  a.tiles = a.tiles_x * ((a.h[0] + kImageTile - 1) / kImageTile);
}

template <class Src>
inline void fill_depth(DepthArgs<Src>& a, const Level* lv, int levels, float* const* inv, float4* const* v,
                       float4* const* p) {
  fill_tiles(a.t, lv, levels);
  for (int l = 0; l < levels; ++l) {
    a.invfx[l] = lv[l].invfx;
    a.invfy[l] = lv[l].invfy;
    a.cx[l] = lv[l].cx;
    a.cy[l] = lv[l].cy;
    a.inv[l] = inv[l];
    a.v[l] = v[l];
    a.p[l] = p[l];
  }
}

}  // namespace yas
