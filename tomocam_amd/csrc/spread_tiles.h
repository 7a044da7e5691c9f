// Which polar points reach which tile of a fine grid: the work of a spreading
// kernel that owns its tiles.  The ray segments that meet a tile are enumerated
// analytically, once per geometry; a tile's points are numbered along its
// segments, and a work item is a tile with a range of its points.
#pragma once

#include <vector>

#include "tc_common.h"

namespace tc {

constexpr int SP_T = 32;  // tile edge (grid points)
// The cells within SP_CENTRE of the grid's centre get points from every ray, and
// the same values again and again (the sample t = 0 of each ray is one point).
// Added one after the other, hundreds in a work item, their rounding is not
// random: a level error of the whole image or PSF (T x of 1454^2 at 720 angles
// against 64 bits: 6.3e-7 with items of 1024 points there, 3.8e-6 with 4096).
// The tiles that hold such cells are cut into items of SP_CENTRE_CHUNK points,
// whose sums the fix-up adds in FP64: 6.4e-8.  (FP32 lists only: FP64 sums need
// no such care, and their angles have no limit that would bound the slots.)
constexpr int SP_CENTRE = 8, SP_CENTRE_CHUNK = 128;

struct TileGeom {
  const double* ax;  // [P] grid steps per sample along x and y
  const double* ay;
  const int2* seg;       // segments of all tiles: angle, first sample | copy << 16
  const int* seg_off;    // their first points' numbers within the tile
  const int* tile_seg;   // [ntiles + 1] first segment of each tile
  int P, N, cidx;        // N samples per ray at t = j - cidx
  int nf, ncols, ntx;    // grid points per axis (periodic), columns kept
  double umax;           // |t step| <= umax
};

struct TileWindow {
  int X0, Y0, X1, Y1;
};

__device__ __forceinline__ TileWindow tile_window(const TileGeom& a, int tile) {
  TileWindow w;
  const int ty = tile / a.ntx;
  const int tx = tile - ty * a.ntx;
  w.X0 = tx * SP_T;
  w.Y0 = ty * SP_T;
  w.X1 = min(w.X0 + SP_T, a.ncols);
  w.Y1 = min(w.Y0 + SP_T, a.nf);
  return w;
}

// grid origin of periodic copy `shift` (0 .. 8, row-major over ky, kx)
__device__ __forceinline__ double2 shift_origin(const TileGeom& a, int shift) {
  const int ky = shift / 3 - 1, kx = shift - (shift / 3) * 3 - 1;
  return make_double2(0.5 * a.nf + kx * (double)a.nf,
                      0.5 * a.nf + ky * (double)a.nf);
}

// First cell of a footprint of W cells and its distance from the point, along
// one axis (fma so that every kernel rounds the coordinate alike).
template <int W, typename T>
__device__ __forceinline__ int first_cell(double origin, double t, double step,
                                          T& frac) {
  const double u = fma(t, step, origin);
  const double c = ceil(u - 0.5 * W);
  frac = (T)(c - u);
  return (int)c;
}

// Rows and columns of wave w's region g (four for each of four waves), of the 16
// regions of 4 rows x 16 columns of a tile: each pair of 4-row bands has one
// region of every wave, and so has each column half over two pairs.  A batch of
// points is a few neighbouring rays, which may cross the tile along a few rows
// or columns; with eight whole rows to a wave, such a batch left most waves
// idle.  (Eight waves of two regions: 15 % slower at 8 x 2048^2, 4 % faster at
// 4 x 256^2.)
constexpr int SP_WAVES = 4, SP_REGIONS = 4;
__device__ __forceinline__ int region_y(int w, int g) {
  return 8 * g + 4 * (((w - g) & 3) >> 1);
}
__device__ __forceinline__ int region_x(int w, int g) {
  return 16 * ((w - g) & 1);
}

constexpr int SP_FIX_HEAVY = 16;

// The lists of one geometry (device) and the work cut from them.
class TileLists {
 public:
  // Points per tile and every tile's segments, for kernel width W (8 or 16);
  // reads the counts back (one synchronisation).  g: ax .. umax filled in.
  void make_segments(const TileGeom& g, int W, hipStream_t stream);
  // The work and fix-up lists for `chunk_max` points per item (FP32: the tiles
  // about the centre at most SP_CENTRE_CHUNK).  Synchronous copies: the caller
  // has no kernel reading the previous lists in flight.
  void make_work(int chunk_max);
  void fill(TileGeom& g) const;  // the list pointers

  // Points per item by rule: a workgroup takes its points 128 at a time, in
  // turn, so a small geometry is cut finely enough to fill the chip (about 768
  // items), down to one batch each; a large one takes 1024 (less fix-up).
  // Spreading and fix-up at 4 x 256^2, 180 angles: 34 us at 512, 22 at 128; at
  // 8 x 512^2, 360 angles: 49 at 512, 36 at 256; at 8 x 2048^2, 1501 angles:
  // 599 at 128, 347 at 512, 321 at 1024.
  int rule_chunk() const;

  int chunk() const { return chunk_; }
  int nwork() const { return nwork_; }
  int nslots() const { return nslots_; }  // scratch tiles of further chunks
  int nfix() const { return nfix_; }
  // the fix-up list starts with the tiles of more than SP_FIX_HEAVY slots
  int nheavy() const { return nheavy_; }
  const int4* work() const { return work_.as<int4>(); }
  const int4* fix() const { return fix_.as<int4>(); }

 private:
  int nwork_ = 0, nslots_ = 0, nfix_ = 0, nheavy_ = 0, chunk_ = 0;
  std::vector<int> counts_;      // polar points per tile
  std::vector<char> centre_;     // tiles cut into items of SP_CENTRE_CHUNK
  std::vector<int> tile_first_;  // first segment of each tile
  DevBuf seg_, seg_off_, tile_seg_;
  // two int4 per item: tile, first point, end point, scratch slot (-1: none);
  // the tile's segment range
  DevBuf work_;
  DevBuf fix_;  // int4: tile, first slot, slot count, 0
};

}  // namespace tc
