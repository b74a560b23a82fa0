// pm_tiles.h -- the 8x8 pixel tiles of the lane renders and their pixel
// output.  Device code and the launchers' grid size.
#pragma once

#include "pm_kernels.h"

namespace pm {

__device__ __forceinline__ void store_pixel(float* rgb, uchar4* u8, size_t o, V3f v, float exposure) {
  if (rgb) {
    rgb[3 * o] = v.x;
    rgb[3 * o + 1] = v.y;
    rgb[3 * o + 2] = v.z;
  }
  if (u8) {
    uchar4 q;
    q.x = tonemap_u8(v.x, exposure);
    q.y = tonemap_u8(v.y, exposure);
    q.z = tonemap_u8(v.z, exposure);
    q.w = 0;
    u8[o] = q;
  }
}

// Workgroups are dispatched to the 8 XCDs of the chip round-robin, and each
// XCD has its own L2.  With tile_regions = rx (1, 2, 4 or 8) the crop's tiles
// are cut into an rx x (8 / rx) grid of regions and workgroup b renders the
// (b / 8)-th tile, in raster order, of region b % 8: each XCD then works on
// one compact part of the frame, and its L2 holds the photons of that part's
// view frustum.  tile_regions = 0 (and raster) renders tile b in raster order.
__host__ __device__ __forceinline__ void tile_regions(const RenderLaunch& r, int tw, int th, bool raster, int& tiles_x,
                                                      int& tiles_y, int& rx, int& ry, int& rw, int& rh) {
  tiles_x = (r.w + tw - 1) / tw;
  tiles_y = (r.h + th - 1) / th;
  rx = raster ? 0 : r.tile_regions;
  ry = 8 / (rx > 0 ? rx : 1);
  rw = (tiles_x + rx - 1) / (rx > 0 ? rx : 1);
  rh = (tiles_y + ry - 1) / ry;
}

// Workgroups of a launch over tw x th pixel tiles.
inline unsigned tile_grid(const RenderLaunch& r, int tw, int th, bool raster) {
  int tiles_x, tiles_y, rx, ry, rw, rh;
  tile_regions(r, tw, th, raster, tiles_x, tiles_y, rx, ry, rw, rh);
  if (rx <= 0) return (unsigned)(tiles_x * tiles_y);
  return 8u * (unsigned)(rw * rh);
}

// Tile (tx, ty) of this workgroup; false when it has none.
__device__ __forceinline__ bool tile_of_block(const RenderLaunch& r, int tw, int th, bool raster, int& tx, int& ty) {
  int tiles_x, tiles_y, rx, ry, rw, rh;
  tile_regions(r, tw, th, raster, tiles_x, tiles_y, rx, ry, rw, rh);
  const int b = (int)blockIdx.x;
  tx = b % tiles_x;
  ty = b / tiles_x;
  if (rx <= 0) return true;
  const int reg = b & 7, slot = b >> 3;
  const int gx = reg % rx, gy = reg / rx;
  // region bounds: the first (tiles mod rx) regions of a row are one wider
  const int x0 = gx * (tiles_x / rx) + min(gx, tiles_x % rx), w = tiles_x / rx + (gx < tiles_x % rx ? 1 : 0);
  const int y0 = gy * (tiles_y / ry) + min(gy, tiles_y % ry), h = tiles_y / ry + (gy < tiles_y % ry ? 1 : 0);
  if (w <= 0 || slot >= w * h) return false;
  tx = x0 + slot % w;
  ty = y0 + slot / w;
  return true;
}

// The lane renders: 8x8 tiles, lane = pixel (lx, ly) of the crop; false when
// it lies outside.
inline unsigned lane_grid(const RenderLaunch& r) { return tile_grid(r, 8, 8, false); }
__device__ __forceinline__ bool lane_tile(const RenderLaunch& r, int lane, int& lx, int& ly) {
  int tx, ty;
  if (!tile_of_block(r, 8, 8, false, tx, ty)) return false;
  lx = tx * 8 + (lane & 7);
  ly = ty * 8 + (lane >> 3);
  return lx < r.w && ly < r.h;
}

}  // namespace pm
