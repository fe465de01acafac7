// A frame's image products, every pyramid level in one launch: intensity
// pyramid with gradients, and the inverse depths, vertices and ICP points of
// a depth image or of a model vertex map (RGBDFusion/src/ImageProc.cu,
// RGBDTracking.cu:60-160).
//
// These images are small (4 us of memory time at 640x480 for all levels
// together), so a launch per level and product, about 4.5 us each back to
// back, was what they cost: 6 launches for an image, 9 for a depth image, 6
// for a model.  Depth and model levels are subsampled, so a pixel of any
// level follows from three pixels of the full image and the levels need no
// order.  The intensity pyramid does: a workgroup takes a 32x32 tile, holds
// the pixels that its levels 1 and 2 need in LDS (49x49, 2.3 times the tile)
// and forms the halo of each level for itself, with the values that the
// level's own workgroups give it.  A frame's calls (conversions, image and
// depth pyramids) went from 54 to 22 us at 640x480 and from 56 to 17 us at
// 160x120, where the four launches left are what the host can enqueue.
#pragma once

#include "yas_tracker_dev.hpp"

namespace yas {

// Sources of the full-size images.
struct SrcF32 {
  const float* p;
  size_t pitch;
  __device__ inline float at(int x, int y) const { return ld(p, pitch, x, y); }
};
struct SrcU16 {  // depth in 1 / scale metres
  const uint16_t* p;
  size_t pitch;
  float scale;
  __device__ inline float at(int x, int y) const {
    return (float)((const uint16_t*)((const char*)p + (size_t)y * pitch))[x] * scale;
  }
};
struct SrcRgb {
  const uint8_t* p;
  size_t pitch;
  int mode;
  __device__ inline float at(int x, int y) const {
    const uint8_t* q = p + (size_t)y * pitch + 3 * x;
    return gray_of(q[0], q[1], q[2], mode);
  }
};

// ------------------------------------------------------------------ intensity
constexpr int kImageTile = 32;    // of the first level, per workgroup
constexpr int kImageLevels = 3;   // levels a launch forms
constexpr int kImageHalo0 = 10;   // first-level pixels before the tile that level 2's gradients reach
constexpr int kImageSpan0 = 49;   // x0 - 10 .. x0 + 38
constexpr int kImageHalo1 = 4, kImageSpan1 = 23;  // x0/2 - 4 .. x0/2 + 18
constexpr int kImageHalo2 = 1, kImageSpan2 = 10;  // x0/4 - 1 .. x0/4 + 8

template <class Src>
struct ImageArgs {
  Src src;               // the first level
  int n;                 // levels, 1..3
  int w[kImageLevels], h[kImageLevels];
  float* out[kImageLevels];  // out[0] null: the first level is not stored and has no gradients here
  float* gx[kImageLevels];   // null: no gradients
  float* gy[kImageLevels];
  int tiles_x, tiles;
};
struct ImageLds {
  float l0[kImageSpan0][kImageSpan0 + 1];
  float l1[kImageSpan1][kImageSpan1 + 1];
  float l2[kImageSpan2][kImageSpan2 + 1];
};

// Level `l`'s pixels of the tile stored from LDS with their gradients;
// (px, py) is the tile's first pixel at that level, `side` its size, `halo`
// the LDS image's pixels before it.
template <int SPAN>
__device__ inline void store_level(const float (&m)[SPAN][SPAN + 1], int halo, int px, int py, int side, int w, int h,
                                   float* out, float* gx, float* gy) {
  for (int i = threadIdx.x; i < side * side; i += blockDim.x) {
    const int lx = i % side, ly = i / side, x = px + lx, y = py + ly;
    if (x >= w || y >= h) continue;
    const int cx = lx + halo, cy = ly + halo;
    const size_t k = (size_t)y * w + x;
    out[k] = m[cy][cx];
    if (!gx) continue;
    float a = 0.0f, b = 0.0f;
    if (!(x < 1 || y < 1 || x > w - 2 || y > h - 2)) {
      a = (m[cy][cx + 1] - m[cy][cx - 1]) * 0.5f;
      b = (m[cy + 1][cx] - m[cy - 1][cx]) * 0.5f;
    }
    gx[k] = a;
    gy[k] = b;
  }
}
// The pixels of the next level that `dst` covers and the image has, from `src`.
template <int S0, int S1>
__device__ inline void down_level(const float (&src)[S0][S0 + 1], int halo0, int px0, int py0, int w0, int h0,
                                  float (&dst)[S1][S1 + 1], int halo1, int px1, int py1, int w1, int h1) {
  for (int i = threadIdx.x; i < S1 * S1; i += blockDim.x) {
    const int cx = i % S1, cy = i / S1, x = px1 - halo1 + cx, y = py1 - halo1 + cy;
    if (x < 0 || y < 0 || x >= w1 || y >= h1) continue;
    dst[cy][cx] = pyrdown_gauss_from(
        [&](int sx, int sy) { return src[sy - py0 + halo0][sx - px0 + halo0]; }, w0, h0, x, y);
  }
}
template <class Src>
__device__ inline void image_tile(const ImageArgs<Src>& a, int tile, ImageLds& S) {
  const int x0 = (tile % a.tiles_x) * kImageTile, y0 = (tile / a.tiles_x) * kImageTile;
  for (int i = threadIdx.x; i < kImageSpan0 * kImageSpan0; i += blockDim.x) {
    const int cx = i % kImageSpan0, cy = i / kImageSpan0, x = x0 - kImageHalo0 + cx, y = y0 - kImageHalo0 + cy;
    if (x >= 0 && y >= 0 && x < a.w[0] && y < a.h[0]) S.l0[cy][cx] = a.src.at(x, y);
  }
  __syncthreads();
  if (a.out[0]) store_level(S.l0, kImageHalo0, x0, y0, kImageTile, a.w[0], a.h[0], a.out[0], a.gx[0], a.gy[0]);
  if (a.n < 2) return;
  const int x1 = x0 / 2, y1 = y0 / 2, x2 = x0 / 4, y2 = y0 / 4;
  down_level(S.l0, kImageHalo0, x0, y0, a.w[0], a.h[0], S.l1, kImageHalo1, x1, y1, a.w[1], a.h[1]);
  __syncthreads();
  store_level(S.l1, kImageHalo1, x1, y1, kImageTile / 2, a.w[1], a.h[1], a.out[1], a.gx[1], a.gy[1]);
  if (a.n < 3) return;
  down_level(S.l1, kImageHalo1, x1, y1, a.w[1], a.h[1], S.l2, kImageHalo2, x2, y2, a.w[2], a.h[2]);
  __syncthreads();
  store_level(S.l2, kImageHalo2, x2, y2, kImageTile / 4, a.w[2], a.h[2], a.out[2], a.gx[2], a.gy[2]);
}

// ------------------------------------------------------------------ depth, model
// The 64x4-pixel tiles of all levels, counted through: level l has tiles
// first[l] .. first[l + 1] - 1.
struct LevelTiles {
  int n;
  int w[kMaxLevels], h[kMaxLevels];
  int first[kMaxLevels + 1];
  // Pixel (x, y) of level l that this thread takes of tile b; false outside.
  __device__ inline bool pixel(int b, int& l, int& x, int& y) const {
    l = 0;
    while (b >= first[l + 1]) ++l;
    b -= first[l];
    const int tx = (w[l] + 63) >> 6;
    x = (b % tx) * 64 + (threadIdx.x & 63);
    y = (b / tx) * 4 + (threadIdx.x >> 6);
    return x < w[l] && y < h[l];
  }
};
inline void fill_tiles(LevelTiles& t, const Level* lv, int n) {
  t.n = n;
  t.first[0] = 0;
  for (int l = 0; l < n; ++l) {
    t.w[l] = lv[l].w;
    t.h[l] = lv[l].h;
    t.first[l + 1] = t.first[l] + ((lv[l].w + 63) / 64) * ((lv[l].h + 3) / 4);
  }
}
// A level above 0 has its last row and column empty; every other pixel is
// one of the level below (so one of level 0).
__device__ inline bool level_has(int l, int x, int y, int w, int h) { return l == 0 || (x < w - 1 && y < h - 1); }

template <class Src>
struct DepthArgs {
  Src src;
  LevelTiles t;
  float invfx[kMaxLevels], invfy[kMaxLevels], cx[kMaxLevels], cy[kMaxLevels];
  float* inv[kMaxLevels];
  float4* v[kMaxLevels];
  float4* p[kMaxLevels];  // ICP points
};
template <class Src>
__device__ inline void depth_tile(const DepthArgs<Src>& a, int b) {
  int l, x, y;
  if (!a.t.pixel(b, l, x, y)) return;
  const int w = a.t.w[l], h = a.t.h[l];
  auto inverse = [&](int i, int j) { return level_has(l, i, j, w, h) ? invdepth_of(a.src.at(i << l, j << l)) : 0.0f; };
  auto vertex = [&](float iv, int i, int j) {
    return vertex_of(iv, i, j, a.invfx[l], a.invfy[l], a.cx[l], a.cy[l], 3.0f);
  };
  const bool nb = x != w - 1 && y != h - 1;
  const float iv = inverse(x, y), ivx = nb ? inverse(x + 1, y) : 0.0f, ivy = nb ? inverse(x, y + 1) : 0.0f;
  const float4 c = vertex(iv, x, y);
  const size_t k = (size_t)y * w + x;
  a.inv[l][k] = iv;
  a.v[l][k] = c;
  store_icp_point(a.p[l], w * h, (int)k, icp_point_of(c, vertex(ivx, x + 1, y), vertex(ivy, x, y + 1), nb));
}

struct ModelArgs {
  const float4* src;
  size_t pitch;
  LevelTiles t;
  float4* v[kMaxLevels];
  float4* p[kMaxLevels];  // ICP points
};
__device__ inline void model_tile(const ModelArgs& a, int b) {
  int l, x, y;
  if (!a.t.pixel(b, l, x, y)) return;
  const int w = a.t.w[l], h = a.t.h[l];
  const float4 none = make_float4(0.f, 0.f, 0.f, -1.f);
  auto vertex = [&](int i, int j) {
    return level_has(l, i, j, w, h)
               ? ((const float4*)((const char*)a.src + (size_t)(j << l) * a.pitch))[(size_t)i << l]
               : none;
  };
  const bool nb = x != w - 1 && y != h - 1;
  const float4 c = vertex(x, y), cx = nb ? vertex(x + 1, y) : none, cy = nb ? vertex(x, y + 1) : none;
  const size_t k = (size_t)y * w + x;
  a.v[l][k] = c;
  store_icp_point(a.p[l], w * h, (int)k, icp_point_of(c, cx, cy, nb));
}

}  // namespace yas
