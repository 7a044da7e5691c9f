// Segment and work lists of tile-owned spreading (spread_tiles.h).
#include <algorithm>

#include "spread_tiles.h"

namespace tc {

// { t : lo < U0 + t a <= hi } intersected into [tlo, thi] (superset bounds)
__device__ __forceinline__ void ray_interval(double a, double U0, double lo,
                                             double hi, double& tlo,
                                             double& thi) {
  if (fabs(a) < 1e-12) {
    if (!(U0 > lo - 1e-9 && U0 <= hi + 1e-9)) {
      tlo = 1e30;
      thi = -1e30;
    }
    return;
  }
  double t1 = (lo - U0) / a, t2 = (hi - U0) / a;
  if (t1 > t2) {
    double q = t1;
    t1 = t2;
    t2 = q;
  }
  tlo = fmax(tlo, t1);
  thi = fmin(thi, t2);
}

// Inclusive prefix sum of one int per thread over a 256-thread block.
__device__ __forceinline__ int block_scan_incl(int v, int* wsum) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int u = __shfl_up(v, d, 64);
    if (lane >= d) v += u;
  }
  if (lane == 63) wsum[wid] = v;
  __syncthreads();
  int off = 0;
  for (int w = 0; w < wid; ++w) off += wsum[w];
  __syncthreads();
  return v + off;
}

// Segments of one tile, counted (FILL false: counts[tile] = points,
// counts[ntiles + tile] = segments) or written to the plan's lists.  Thread t
// examines angles t, t + 256, ... of each periodic copy, in turn; a segment is
// trimmed to the samples whose footprints really meet the tile.  The order
// (copy, then a block-scanned order of the angles) is fixed, so every call of
// the geometry adds a tile's points in the same order.
template <int W, bool FILL>
__global__ void __launch_bounds__(256)
spread_segments_kernel(TileGeom a, int* counts, int2* seg, int* seg_off) {
  __shared__ int wsum[4];
  __shared__ int carry[2];
  const int tile = blockIdx.x, tid = threadIdx.x;
  const TileWindow w = tile_window(a, tile);
  const double lox = w.X0 - 0.5 * W, hix = w.X1 - 1 + 0.5 * W;
  const double loy = w.Y0 - 0.5 * W, hiy = w.Y1 - 1 + 0.5 * W;
  const int s0 = FILL ? a.tile_seg[tile] : 0;
  int nseg = 0, npts = 0;
  for (int shift = 0; shift < 9; ++shift) {
    const double2 o = shift_origin(a, shift);
    if (o.x + a.umax <= lox || o.x - a.umax > hix || o.y + a.umax <= loy ||
        o.y - a.umax > hiy)
      continue;
    for (int p0 = 0; p0 < a.P; p0 += 256) {
      const int p = p0 + tid;
      int jl = 1, jh = 0;
      if (p < a.P) {
        const double ax = a.ax[p], ay = a.ay[p];
        double tlo = -1e30, thi = 1e30;
        ray_interval(ax, o.x, lox, hix, tlo, thi);
        ray_interval(ay, o.y, loy, hiy, tlo, thi);
        if (tlo <= thi) {
          tlo = fmax(tlo, -(double)a.N - 2.0);
          thi = fmin(thi, (double)a.N + 2.0);
          jl = max(0, (int)floor(tlo) + a.cidx - 1);
          jh = min(a.N - 1, (int)ceil(thi) + a.cidx + 1);
          auto meets = [&](int j) {
            double f;
            const double t = (double)(j - a.cidx);
            const int lx = first_cell<W>(o.x, t, ax, f);
            const int ly = first_cell<W>(o.y, t, ay, f);
            return lx < w.X1 && lx + W > w.X0 && ly < w.Y1 &&
                   ly + W > w.Y0;
          };
          while (jl <= jh && !meets(jl)) ++jl;
          while (jl <= jh && !meets(jh)) --jh;
        }
      }
      const int len = max(0, jh - jl + 1), has = len > 0;
      const int iseg = block_scan_incl(has, wsum);
      const int ipts = block_scan_incl(len, wsum);
      if (FILL && has) {
        seg[s0 + nseg + iseg - 1] = make_int2(p, jl | (shift << 16));
        seg_off[s0 + nseg + iseg - 1] = npts + ipts - len;
      }
      if (tid == 255) {
        carry[0] = iseg;
        carry[1] = ipts;
      }
      __syncthreads();
      nseg += carry[0];
      npts += carry[1];
      __syncthreads();
    }
  }
  if (!FILL && tid == 0) {
    counts[tile] = npts;
    counts[gridDim.x + tile] = nseg;
  }
}

int TileLists::rule_chunk() const {
  long total = 0;
  for (int c : counts_) total += c;
  int chunk = 128;
  while (chunk < 1024 && total > 768L * chunk) chunk *= 2;
  return chunk;
}

void TileLists::fill(TileGeom& g) const {
  g.seg = seg_.as<int2>();
  g.seg_off = seg_off_.as<int>();
  g.tile_seg = tile_seg_.as<int>();
}

void TileLists::make_segments(const TileGeom& geom, int W, hipStream_t stream) {
  ArenaPause no_arena;  // the plan's lists, offsets filled synchronously
  TC_REQUIRE(geom.N < 65536, "spreading: too many samples per ray");
  TileGeom g = geom;
  const int ntiles = g.ntx * (int)cdiv(g.nf, SP_T);
  auto count = W == 8 ? spread_segments_kernel<8, false>
                      : spread_segments_kernel<16, false>;
  auto list = W == 8 ? spread_segments_kernel<8, true>
                     : spread_segments_kernel<16, true>;
  DevBuf dcounts(sizeof(int) * 2 * ntiles);
  hipLaunchKernelGGL(count, dim3(ntiles), dim3(256), 0, stream, g,
                     dcounts.as<int>(), nullptr, nullptr);
  TC_HIP(hipGetLastError());
  std::vector<int> h(2 * (size_t)ntiles);
  TC_HIP(hipMemcpyAsync(h.data(), dcounts.as<void>(), sizeof(int) * h.size(),
                        hipMemcpyDeviceToHost, stream));
  TC_HIP(hipStreamSynchronize(stream));
  counts_.assign(h.begin(), h.begin() + ntiles);
  centre_.assign(ntiles, 0);
  if (W == 8) {
    const int lo = std::max(0, (g.nf / 2 - SP_CENTRE) / SP_T);
    const int hi = (g.nf / 2 + SP_CENTRE) / SP_T;
    for (int ty = lo; ty <= std::min(hi, ntiles / g.ntx - 1); ++ty)
      for (int tx = lo; tx <= std::min(hi, g.ntx - 1); ++tx)
        centre_[ty * g.ntx + tx] = 1;
  }
  tile_first_.assign(ntiles + 1, 0);
  for (int t = 0; t < ntiles; ++t)
    tile_first_[t + 1] = tile_first_[t] + h[ntiles + t];
  tile_seg_.alloc(sizeof(int) * tile_first_.size());
  TC_HIP(hipMemcpy(tile_seg_.as<void>(), tile_first_.data(),
                   sizeof(int) * tile_first_.size(), hipMemcpyHostToDevice));
  const size_t nseg = std::max(1, tile_first_[ntiles]);
  seg_.alloc(sizeof(int2) * nseg);
  seg_off_.alloc(sizeof(int) * nseg);
  fill(g);
  hipLaunchKernelGGL(list, dim3(ntiles), dim3(256), 0, stream, g, nullptr,
                     seg_.as<int2>(), seg_off_.as<int>());
  TC_HIP(hipGetLastError());
}

// The work and fix-up lists for `chunk_max` points per item, uploaded to the
// plan's buffers (synchronous copies: the caller has no kernel reading the
// previous lists in flight).
void TileLists::make_work(int chunk_max) {
  ArenaPause no_arena;  // the plan's work lists, filled synchronously
  const int ntiles = (int)counts_.size();
  std::vector<int4> work, fix;
  int slot = 0;
  for (int t = 0; t < ntiles; ++t) {
    const int c = counts_[t];
    const int chunk =
        centre_[t] ? std::min(chunk_max, SP_CENTRE_CHUNK) : chunk_max;
    const int nch = std::max(1, (c + chunk - 1) / chunk);
    work.push_back(make_int4(t, 0, std::min(c, chunk), -1));
    if (nch > 1) {
      fix.push_back(make_int4(t, slot, nch - 1, 0));
      for (int k = 1; k < nch; ++k)
        work.push_back(make_int4(t, k * chunk, std::min(c, (k + 1) * chunk),
                                 slot++));
    }
  }
  // Heaviest items first: a workgroup's time grows with its points, and
  // workgroups start in block order, so the long ones must not be last
  // (16 x 2908^2 at 1501 angles: 28.6 -> 19.9 ms per backprojection).
  // Block b reads item xcd_remap(b) (each XCD takes a contiguous range of
  // the list), so rank b of the sorted order goes to index xcd_remap(b).
  // Each item writes its own tile or slot, and the fix-up adds slots in
  // slot order, so the result does not depend on the order.
  {
    std::vector<int4> byw(work);
    std::stable_sort(byw.begin(), byw.end(), [](const int4& x, const int4& y) {
      return x.z - x.y > y.z - y.y;
    });
    const int n = (int)byw.size();
    const int q = n >> 3, rmd = n & 7;
    for (int b = 0; b < n; ++b) {
      const int x = b & 7, t = b >> 3;
      work[x * q + (x < rmd ? x : rmd) + t] = byw[b];
    }
  }
  // a fix-up's time grows with the slots of its tile
  std::stable_sort(fix.begin(), fix.end(), [](const int4& x, const int4& y) {
    return x.z > y.z;
  });
  // each item with its tile's range of segments
  std::vector<int4> items;
  items.reserve(2 * work.size());
  for (const int4& x : work) {
    items.push_back(x);
    items.push_back(make_int4(tile_first_[x.x], tile_first_[x.x + 1], 0, 0));
  }
  nwork_ = (int)work.size();
  nslots_ = slot;
  nfix_ = (int)fix.size();
  nheavy_ = 0;
  while (nheavy_ < nfix_ && fix[nheavy_].z > SP_FIX_HEAVY) ++nheavy_;
  chunk_ = chunk_max;
  work_.alloc(sizeof(int4) * items.size());
  TC_HIP(hipMemcpy(work_.as<void>(), items.data(), sizeof(int4) * items.size(),
                   hipMemcpyHostToDevice));
  if (nfix_) {
    fix_.alloc(sizeof(int4) * nfix_);
    TC_HIP(hipMemcpy(fix_.as<void>(), fix.data(), sizeof(int4) * nfix_,
                     hipMemcpyHostToDevice));
  }
}

}  // namespace tc
