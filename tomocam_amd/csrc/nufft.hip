// Polar-grid NUFFT (tile-owned spreading on the matrix cores, gather
// interpolation), ray DFT (direct or Bluestein) and the projectors built on them.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <mutex>
#include <tuple>

#include "fft_device.h"
#include "fft_ops.h"
#include "lds_launch.h"
#include "nufft.h"

namespace tc {

// ---------------------------------------------------------------------------
// kernel function and host-side correction factors
// ---------------------------------------------------------------------------

// exp(beta (sqrt(1 - z^2) - 1)) on |z| <= 1, else 0, with hardware sqrt, rcp
// and exp2 (about 1 ulp each).
//
// Type 1 takes the exponent as -beta z^2 / (1 + sqrt(1 - z^2)): the difference
// sqrt - 1 carries the root's rounding, times beta, into the weights near the
// kernel's centre, a level error of up to 6e-7 of an image.  Type 2 keeps the
// difference form.  The other would be more exact there too (the gradient of
// 1/2 |P x - y|^2 at 8 x 512^2 is 2.3e-5 off 64 bits, 3.5e-6 with it), but that
// gradient amplifies any change of P x's level, and would move by more than 2e-5.
__device__ __forceinline__ float es_kernel(float z, float beta) {
  const float s = fmaf(-z, z, 1.0f);
  const float r = __builtin_amdgcn_sqrtf(fmaxf(s, 0.f)) + 1.0f;
  const float e = __builtin_amdgcn_exp2f(-1.44269504088896341f * beta *
                                         (z * z) * __builtin_amdgcn_rcpf(r));
  return s >= 0.f ? e : 0.f;
}
__device__ __forceinline__ float es_kernel_diff(float z, float beta) {
  const float s = 1.0f - z * z;
  const float e = __builtin_amdgcn_exp2f(
      beta * 1.44269504088896341f *
      (__builtin_amdgcn_sqrtf(fmaxf(s, 0.f)) - 1.0f));
  return s >= 0.f ? e : 0.f;
}

// Gauss-Legendre nodes/weights on [-1, 1] (Newton iteration on P_n).
static void gauss_legendre(int n, std::vector<double>& x, std::vector<double>& w) {
  x.assign(n, 0.0);
  w.assign(n, 0.0);
  for (int i = 0; i < n; ++i) {
    double z = std::cos(M_PI * (i + 0.75) / (n + 0.5));
    double pp = 1.0;
    for (int it = 0; it < 100; ++it) {
      double p1 = 1.0, p2 = 0.0;
      for (int j = 1; j <= n; ++j) {
        double p3 = p2;
        p2 = p1;
        p1 = ((2.0 * j - 1.0) * z * p2 - (j - 1.0) * p3) / j;
      }
      pp = n * (z * p1 - p2) / (z * z - 1.0);
      double z1 = z;
      z = z1 - p1 / pp;
      if (std::fabs(z - z1) < 1e-15) {
        p1 = 1.0;
        p2 = 0.0;
        for (int j = 1; j <= n; ++j) {
          double p3 = p2;
          p2 = p1;
          p1 = ((2.0 * j - 1.0) * z * p2 - (j - 1.0) * p3) / j;
        }
        pp = n * (z * p1 - p2) / (z * z - 1.0);
        break;
      }
    }
    x[i] = z;
    w[i] = 2.0 / ((1.0 - z * z) * pp * pp);
  }
}

// ---------------------------------------------------------------------------
// spreading (type 1): each workgroup owns a T x T tile of the fine grid and
// adds every polar point whose kernel footprint meets it, from the geometry's
// segment lists (spread_tiles.h): no sorting and no global atomics.
// ---------------------------------------------------------------------------

struct SpreadArgs {
  TileGeom g;       // columns 0 .. g.ncols - 1 of the grid
  const float2* c;  // [nsl][P][nh]: values at t = 0 .. nh - 1, t < 0 conjugate
  float2* fine;     // [nsl][half_grid_size(g.nf)]
  int nsl, nh;
  float beta;
};

// One workgroup per (work item, group of SB slices): the points [f0, f1) of
// its tile as a matrix product on the matrix cores.  The tile is 16 regions
// of 4 rows x 16 columns, four to a wave.  For a region, a slice pair and
// four points, v_mfma_f32_16x16x4 multiplies
//   A[4 r + e][k] = wy_k(row r) c_k(e)   (e: Re, Im of either slice)
//   B[k][x]       = wx_k(column x)
// so the region's cells are accumulated in FP32 registers: lane (r, x) holds
// the four values of cell (r, x).  Points are prepared in batches of SP_BATCH
// (one thread a point: footprint cell, 8 + 8 kernel weights and the slices'
// values, to LDS); each wave then lists the points that meet a region, in
// point order, and takes them four at a time.  Weights outside the footprint
// are zero.  Every cell adds its points in list order: deterministic.
//
// The former kernel added points to LDS cells (read, add, write of 8 bytes per
// cell, slice and point), about 615 SIMD cycles a point for four slices; here
// a point costs 16.6 % of 16 regions x 32 cycles for two slices.
// 8 x 2048^2 at 1501 angles (4374^2 grid, 613 MB of half grids): 0.34 ms, of
// which writing takes 0.13 at the rate of a large copy.  Four waves a SIMD: with
// three (144 registers) 0.38 ms, five spill (0.36 ms).
constexpr int SP_BATCH = 128;

using f32x4 = __attribute__((__vector_size__(4 * sizeof(float)))) float;

template <int SB>
__global__ void __launch_bounds__(64 * SP_WAVES, 4)
spread_kernel(SpreadArgs a, const int4* __restrict__ work, float2* scratch) {
  constexpr int Q = SB / 2;  // slice pairs
  // rows padded so that one thread a row writes 16 bytes without conflicts
  constexpr int CS = Q == 1 ? 4 : 4 * Q + 4;
  // x weights at 4 .. 11 and y weights at 16 .. 23, a zero on either side of
  // each run: a cell outside the footprint reads one of those
  __shared__ alignas(16) float pt_w[SP_BATCH][28];
  // [Re, Im of even slices, Re, Im of odd slices][slice pair]
  __shared__ alignas(16) float pt_c[SP_BATCH][CS];
  __shared__ short2 pt_geo[SP_BATCH];  // (index | l0x << 8, l0y)
  __shared__ int wlist[SP_WAVES][SP_BATCH + 12];
  __shared__ int sg_off[SP_BATCH + 1];
  __shared__ int2 sg[SP_BATCH];
  __shared__ int sg_first;
  static_assert(SP_T == 32, "four 8-row bands per tile");
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lm = lane & 15, lk = lane >> 4;
  const int wi = xcd_remap(blockIdx.x, gridDim.x);
  const int4 item = work[2 * wi];
  const int4 segs = work[2 * wi + 1];  // the tile's segments [x, y)
  const int s0 = blockIdx.y * SB;
  const int ns = min(SB, a.nsl - s0);
  const TileWindow w = tile_window(a.g, item.x);
  const long sstride = (long)a.g.P * a.nh;
  const int seg1 = segs.y;
  f32x4 acc[SP_REGIONS][Q];
#pragma unroll
  for (int g = 0; g < SP_REGIONS; ++g)
#pragma unroll
    for (int q = 0; q < Q; ++q) acc[g][q] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (tid < SP_BATCH) {
    pt_w[tid][3] = pt_w[tid][12] = 0.f;
    pt_w[tid][15] = pt_w[tid][24] = 0.f;
  }
  int seg = segs.x;
  if (item.y > 0) {
    // the segment that holds point f0 (offsets ascend from 0 at segs.x)
    for (int i = seg + tid; i < seg1; i += 64 * SP_WAVES) {
      const int nxt = i + 1 < seg1 ? a.g.seg_off[i + 1] : 0x7fffffff;
      if (a.g.seg_off[i] <= item.y && item.y < nxt) sg_first = i;
    }
    __syncthreads();
    seg = sg_first;
  }
  // half 0 prepares x (and even slices) of point `pt`, half 1 y (odd slices)
  const int pt = tid & (SP_BATCH - 1);
  const int half = __builtin_amdgcn_readfirstlane(tid / SP_BATCH);
  for (int fb0 = item.y; fb0 < item.z; fb0 += SP_BATCH) {
    const int nb = min(SP_BATCH, item.z - fb0);
    // the batch's segments: every segment has a point, so at most nb of them
    if (tid <= SP_BATCH) {
      const int i = seg + tid;
      sg_off[tid] = i < seg1 ? a.g.seg_off[i] : 0x7fffffff;
      if (tid < SP_BATCH) sg[tid] = i < seg1 ? a.g.seg[i] : make_int2(0, 0);
    }
    __syncthreads();
    auto segment_of = [&](int f, int n) {  // sg_off[lo] <= f < sg_off[lo + 1]
      int lo = 0, hi = n;
      while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (sg_off[mid] <= f) lo = mid;
        else hi = mid;
      }
      return lo;
    };
    if (pt < nb) {
      const int f = fb0 + pt;
      const int lo = segment_of(f, SP_BATCH);
      const int p = sg[lo].x, js = sg[lo].y;
      const int t = (js & 0xffff) + (f - sg_off[lo]) - a.g.cidx;
      const float2* cp =
          a.c + (long)(s0 + half) * sstride + (long)p * a.nh + abs(t);
      float2 cv[Q];
#pragma unroll
      for (int q = 0; q < Q; ++q)
        cv[q] = 2 * q + half < ns ? cp[2 * q * sstride] : make_float2(0.f, 0.f);
      const double2 o = shift_origin(a.g, js >> 16);
      float frac;
      const int l0 = first_cell<NUFFT_W>(half ? o.y : o.x, (double)t,
                                         half ? a.g.ay[p] : a.g.ax[p], frac) -
                     (half ? w.Y0 : w.X0);  // -7 .. 31
      if (half)
        pt_geo[pt].y = (short)l0;
      else
        pt_geo[pt].x = (short)(pt | (l0 << 8));
      float wt[NUFFT_W];
#pragma unroll
      for (int m = 0; m < NUFFT_W; ++m)
        wt[m] = es_kernel((frac + (float)m) * (2.0f / NUFFT_W), a.beta);
#pragma unroll
      for (int m = 0; m < NUFFT_W; ++m) pt_w[pt][12 * half + 4 + m] = wt[m];
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        pt_c[pt][(2 * half) * Q + q] = cv[q].x;
        pt_c[pt][(2 * half + 1) * Q + q] = t < 0 ? -cv[q].y : cv[q].y;
      }
      // the segment of the next batch's first point
      if (tid == nb - 1) sg_first = seg + segment_of(fb0 + nb, SP_BATCH + 1);
    } else if (half == 0) {
      pt_geo[pt] = make_short2((short)(pt | (100 << 8)), 100);  // no region
    }
    __syncthreads();
    seg = sg_first;
#pragma unroll
    for (int g = 0; g < SP_REGIONS; ++g) {
      const int ry = region_y(wave, g), rx = region_x(wave, g);
      // points whose footprints meet the region, in point order: index and
      // footprint origin in the region, plus 8
      int cnt = 0;
#pragma unroll
      for (int c = 0; c < SP_BATCH / 64; ++c) {
        const short2 e = pt_geo[c * 64 + lane];
        const int dx = (e.x >> 8) - rx, dy = e.y - ry;
        const bool hit = dx > -NUFFT_W && dx < 16 && dy > -NUFFT_W && dy < 4;
        const unsigned long long bal = __ballot(hit);
        const int pos =
            cnt + __builtin_amdgcn_mbcnt_hi((unsigned)(bal >> 32),
                                            __builtin_amdgcn_mbcnt_lo(
                                                (unsigned)bal, 0u));
        if (hit)
          wlist[wave][pos] = (e.x & 0xff) | (dx + 8) << 8 | (dy + 8) << 16;
        cnt += __popcll(bal);
      }
      if (cnt == 0) continue;
      // the steps and look-ahead past the end take a point of the batch with
      // its footprint out of reach
      if (lane < 12) wlist[wave][cnt + lane] = 0xffff00;
      __builtin_amdgcn_wave_barrier();
      // Steps of four points; the next step's weights and values and the list
      // entries of the one after it are read from LDS while this one's
      // products run.
      struct Step {
        float wx, wy, c[Q];
      };
      auto fetch = [&](int e) {
        Step t;
        const int i = e & 0xff;
        const int dx = min(max(lm + 8 - ((e >> 8) & 0xff), -1), 8);
        const int dy = min(max((lm >> 2) + 8 - ((e >> 16) & 0xff), -1), 8);
        t.wx = pt_w[i][4 + dx];
        t.wy = pt_w[i][16 + dy];
#pragma unroll
        for (int q = 0; q < Q; ++q) t.c[q] = pt_c[i][(lm & 3) * Q + q];
        return t;
      };
      Step cur = fetch(wlist[wave][lk]);
      int e1 = wlist[wave][4 + lk];
      for (int k0 = 0; k0 < cnt; k0 += 4) {
        const Step nxt = fetch(e1);
        e1 = wlist[wave][k0 + 8 + lk];
#pragma unroll
        for (int q = 0; q < Q; ++q)
          acc[g][q] = __builtin_amdgcn_mfma_f32_16x16x4f32(
              cur.wy * cur.c[q], cur.wx, acc[g][q], 0, 0, 0);
        cur = nxt;
      }
    }
    __syncthreads();  // the batch buffers are rewritten next
  }
  if (item.w >= 0) {
    float2* dst = scratch + ((long)item.w * gridDim.y + blockIdx.y) *
                                (SB * SP_T * SP_T);
#pragma unroll
    for (int g = 0; g < SP_REGIONS; ++g) {
      const int ly = region_y(wave, g) + lk, lx = region_x(wave, g) + lm;
#pragma unroll
      for (int s = 0; s < SB; ++s)
        dst[(s * SP_T + ly) * SP_T + lx] =
            make_float2(acc[g][s >> 1][2 * (s & 1)],
                        acc[g][s >> 1][2 * (s & 1) + 1]);
    }
    return;
  }
  // A region is four column blocks of four rows, 512 bytes a slice in the
  // grid's order, but the lanes hold it row by row.  Two slices at a time go
  // through LDS, so that sixteen lanes write 256 adjacent bytes (straight from
  // the lanes, 32 at a time: 4 x 256^2 at 180 angles 15.4 -> 14.8 us, 8 x 2048^2
  // 344 -> 340 us).
  // The batches' last barrier is behind every wave; without a batch the zeros
  // written above and here are the same.
  float2* stage = reinterpret_cast<float2*>(&pt_w[0][0]) + 128 * wave;
  const int put = (lm >> 2) * 16 + lk * 4 + (lm & 3);
  const int j = lane & 31, hs = lane >> 5;
#pragma unroll
  for (int g = 0; g < SP_REGIONS; ++g) {
    const int gy = w.Y0 + region_y(wave, g) + ((j >> 1) & 3);
    const int gx = w.X0 + region_x(wave, g) + 4 * (j >> 3) + 2 * (j & 1);
    const bool in = gy < w.Y1 && gx < w.X1;  // column w.X1 may be padding
    float2* o = a.fine + (s0 + hs) * half_grid_size(a.g.nf) +
                (in ? half_at(a.g.nf, gy, gx) : 0u);
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      stage[put] = make_float2(acc[g][q][0], acc[g][q][1]);
      stage[64 + put] = make_float2(acc[g][q][2], acc[g][q][3]);
      __builtin_amdgcn_wave_barrier();
      const float4 val = *reinterpret_cast<const float4*>(stage + 2 * lane);
      __builtin_amdgcn_wave_barrier();
      if (in && 2 * q + hs < ns)
        *reinterpret_cast<float4*>(o + 2 * q * half_grid_size(a.g.nf)) = val;
    }
  }
}

// Adds the scratch slots of multi-chunk tiles into the fine grid, in slot
// order (deterministic).  sb: slices per group of the spreading launch.
// blockIdx.z picks a slice of the group.  A thread sums four cells over the
// slots, four slots at a time (16 loads in flight); of the first nheavy tiles,
// whose slots would be a long chain, one cell and sixteen slots at a time, four
// workgroups a tile.  (All tiles that way: 22 instead of 11 us at 8 x 512^2,
// where most tiles have few slots; none: 32 instead of 19 us at 8 x 2048^2,
// whose centre has 211 slots, 14 instead of 12 at 8 x 512^2.)  The order per
// cell is slot order.  The sums are FP64: the centre's cells add a value of the
// same sign from every ray over many slots, and their rounding is a level error
// of the whole image.
template <int PER, int U>
__device__ __forceinline__ void spread_fixup(const SpreadArgs& a, int4 f, int s,
                                             const float2* base,
                                             long slot_stride, int first) {
  const TileWindow w = tile_window(a.g, f.x);
  base += first;
  double2 sum[PER];
#pragma unroll
  for (int e = 0; e < PER; ++e) sum[e] = make_double2(0.0, 0.0);
  int k = 0;
  for (; k + U <= f.z; k += U) {
    float2 q[U][PER];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < PER; ++e)
        q[u][e] = base[(long)(k + u) * slot_stride + 256 * e];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < PER; ++e) {
        sum[e].x += q[u][e].x;
        sum[e].y += q[u][e].y;
      }
  }
  for (; k < f.z; ++k) {
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const float2 q = base[(long)k * slot_stride + 256 * e];
      sum[e].x += q.x;
      sum[e].y += q.y;
    }
  }
#pragma unroll
  for (int e = 0; e < PER; ++e) {
    const int cell = first + 256 * e;
    const int ly = cell / SP_T, lx = cell - ly * SP_T;
    if (w.Y0 + ly < w.Y1 && w.X0 + lx < w.X1) {
      float2* o = a.fine + s * half_grid_size(a.g.nf) +
                  half_at(a.g.nf, w.Y0 + ly, w.X0 + lx);
      const float2 cur = *o;
      *o = make_float2((float)(cur.x + sum[e].x), (float)(cur.y + sum[e].y));
    }
  }
}

__global__ void __launch_bounds__(256)
spread_fixup_kernel(SpreadArgs a, const int4* __restrict__ fix, int nheavy,
                    const float2* __restrict__ scratch, int sb) {
  static_assert(SP_T * SP_T == 4 * 256, "four cells a thread");
  const int s = blockIdx.y * sb + blockIdx.z;
  if (s >= a.nsl) return;
  const int b = blockIdx.x;
  const bool heavy = b < 4 * nheavy;
  const int4 f = fix[heavy ? b / 4 : b - 3 * nheavy];
  const long slot_stride = (long)gridDim.y * sb * (SP_T * SP_T);
  const float2* base =
      scratch + (long)f.y * slot_stride + (long)s * (SP_T * SP_T);
  if (heavy)
    spread_fixup<1, 16>(a, f, s, base, slot_stride,
                        256 * (b & 3) + (int)threadIdx.x);
  else
    spread_fixup<4, 4>(a, f, s, base, slot_stride, threadIdx.x);
}

// ---------------------------------------------------------------------------
// interpolation (type 2): eight lanes per polar point, all slices of a batch
// ---------------------------------------------------------------------------

struct InterpArgs {
  const float2* fine;  // [nsl][half_grid_size(nf)]
  float2* c;           // [nsl][P][nh]
  const double* ax;
  const double* ay;
  int P, N, nh, nf, nsl;
  float beta;
};

// Samples t and -t of a ray are conjugate (the image is real), so each pair is
// evaluated once, at whichever of the two lies in the stored half of the grid
// (columns up to nf/2); a footprint column past either end of that half is
// read at its mirror image, conjugated.
//
// Eight lanes take a point.  The grid stores HG_B = 4 columns a block, four
// rows of a block in 128 bytes, and a footprint's 8 columns lie in three
// blocks: lane (r, c) = (b >> 1, b & 1) reads columns 2 c, 2 c + 1 of every
// block in rows r and r + 4, six 16-byte loads a slice, each covering 128
// adjacent bytes a point (weights past the footprint are zero).  The loads
// are bound by the cache lines they touch, about 10 a point and slice; one
// column a lane, row by row, touched about 22 (8 x 1024^2 at 720 angles:
// 117 -> 91 us; 8 x 512^2 at 360: 41 -> 27 us).  Where the three blocks reach
// past the stored half (near columns 0 and nf/2) the wave takes that form: lane
// b reads footprint column b of every row, or its mirror image.
//
// The eight lanes' sums are then added across the group for eight slices at
// once by a transposing butterfly (exchange halves with lanes b^4, b^2, b^1:
// 14 shuffles per eight slices), after which lane b holds slice b of the chunk
// and writes it.  The summation order is fixed by the geometry, so results are
// deterministic.
__device__ __forceinline__ float2 shfl_xor2(float2 v, int m) {
  return make_float2(__shfl_xor(v.x, m, 8), __shfl_xor(v.y, m, 8));
}

// Sum over the group's lanes of a lane's part(q) for slices q = 0 .. 7: lane b
// gets slice b's.  Each exchange halves the slices a lane stands for; they are
// taken in the order that lets every exchange happen as soon as it can, so
// that few partial sums are held.
template <int M, class F>
__device__ __forceinline__ float2 group_sum(const F& part, int b, int q) {
  if constexpr (M == 0) {
    return part(q);
  } else {
    const float2 lo = group_sum<M == 4 ? 0 : 2 * M>(part, b, q);
    const float2 hi = group_sum<M == 4 ? 0 : 2 * M>(part, b, q + M);
    const bool up = (b & M) != 0;
    const float2 keep = up ? hi : lo, got = shfl_xor2(up ? lo : hi, M);
    return make_float2(keep.x + got.x, keep.y + got.y);
  }
}

__global__ void __launch_bounds__(256) interp_kernel(InterpArgs a) {
  // each XCD takes adjacent rays, whose footprints overlap in its L2
  const long gid =
      (long)xcd_remap(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  const long pt = gid >> 3;
  const int b = (int)(gid & 7);
  // groups of eight are aligned to eight lanes: a group is all in or out
  if (pt >= (long)a.P * a.nh) return;
  const int p = (int)(pt / a.nh);
  const int m = (int)(pt - (long)p * a.nh);
  const double ax = a.ax[p];
  const double t = ax > 0.0 ? -(double)m : (double)m;
  float fx, fy;
  const int l0x = first_cell<NUFFT_W>(0.5 * a.nf, t, ax, fx);
  const int l0y = first_cell<NUFFT_W>(0.5 * a.nf, t, a.ay[p], fy);
  const float wxb = es_kernel_diff((fx + (float)b) * (2.0f / NUFFT_W), a.beta);
  const float wyb = es_kernel_diff((fy + (float)b) * (2.0f / NUFFT_W), a.beta);
  // conjugated where t < 0 was evaluated for t > 0; the sample at the ray's
  // end of an even N is halved (RayArgs)
  const float end = 2 * m == a.N ? 0.5f : 1.0f;
  const float endi = t < 0.0 ? -end : end;
  const long plane = half_grid_size(a.nf);
  const long cplane = (long)a.P * a.nh;
  const int x0 = l0x & ~(HG_B - 1);
  if (!__any(l0x < 0 || x0 + 3 * HG_B > a.nf / 2 + 1)) {
    const int r0 = b >> 1, c0 = 2 * (b & 1);
    float wx[3][2], wy[2];
    unsigned off[2];
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int f = x0 + HG_B * j + c0 + e - l0x;  // footprint column
        const float w = __shfl(wxb, f & 7, 8);
        wx[j][e] = f >= 0 && f < NUFFT_W ? w : 0.f;
      }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      wy[h] = __shfl(wyb, r0 + 4 * h, 8);
      int qy = l0y + r0 + 4 * h;
      qy += qy < 0 ? a.nf : (qy >= a.nf ? -a.nf : 0);
      off[h] = half_at(a.nf, qy, x0) + c0;
    }
    for (int s0 = 0; s0 < a.nsl; s0 += 8) {
      auto part = [&](int q) {
        const float2* g = a.fine + (long)(s0 + q) * plane;
        float4 val[2][3];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int j = 0; j < 3; ++j)
            val[h][j] = *reinterpret_cast<const float4*>(
                g + (long)j * HG_B * a.nf + off[h]);
        float2 sum[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          sum[h] = make_float2(0.f, 0.f);
#pragma unroll
          for (int j = 0; j < 3; ++j) {
            sum[h].x = fmaf(val[h][j].x, wx[j][0], sum[h].x);
            sum[h].y = fmaf(val[h][j].y, wx[j][0], sum[h].y);
            sum[h].x = fmaf(val[h][j].z, wx[j][1], sum[h].x);
            sum[h].y = fmaf(val[h][j].w, wx[j][1], sum[h].y);
          }
        }
        return make_float2(fmaf(wy[1], sum[1].x, wy[0] * sum[0].x),
                           fmaf(wy[1], sum[1].y, wy[0] * sum[0].y));
      };
      // whole chunks without a branch a slice, so that loads of several slices
      // are in flight
      const float2 v =
          s0 + 8 <= a.nsl
              ? group_sum<1>(part, b, 0)
              : group_sum<1>(
                    [&](int q) {
                      return s0 + q < a.nsl ? part(q) : make_float2(0.f, 0.f);
                    },
                    b, 0);
      if (s0 + b < a.nsl)
        a.c[(long)(s0 + b) * cplane + pt] = make_float2(end * v.x, endi * v.y);
    }
    return;
  }
  int qx = l0x + b;
  qx += qx < 0 ? a.nf : (qx >= a.nf ? -a.nf : 0);
  const bool mirror = 2 * qx > a.nf;
  if (mirror) qx = a.nf - qx;
  float wy[NUFFT_W];
  unsigned roff[NUFFT_W];
#pragma unroll
  for (int r = 0; r < NUFFT_W; ++r) {
    wy[r] = __shfl(wyb, r, 8);
    int qy = l0y + r;
    qy += qy < 0 ? a.nf : (qy >= a.nf ? -a.nf : 0);
    if (mirror && qy > 0) qy = a.nf - qy;
    roff[r] = half_at(a.nf, qy, qx);
  }
  const float flip = mirror ? -wxb : wxb;
  // a slice at a time: few waves come here, and must not cost the others
  // registers
#pragma unroll 1
  for (int s = 0; s < a.nsl; ++s) {
    const float2* g = a.fine + (long)s * plane;
    float2 val[NUFFT_W];
#pragma unroll
    for (int r = 0; r < NUFFT_W; ++r) val[r] = g[roff[r]];
    float2 acc = make_float2(0.f, 0.f);
#pragma unroll
    for (int r = 0; r < NUFFT_W; ++r) {
      acc.x = fmaf(val[r].x, wy[r], acc.x);
      acc.y = fmaf(val[r].y, wy[r], acc.y);
    }
    {
      // no contraction: every lane holds the same sum, whichever stores it
#pragma clang fp contract(off)
      acc = make_float2(acc.x * wxb, acc.y * flip);
#pragma unroll
      for (int k = 4; k > 0; k >>= 1) {
        const float2 got = shfl_xor2(acc, k);
        acc = make_float2(acc.x + got.x, acc.y + got.y);
      }
    }
    if (b == (s & 7))
      a.c[(long)s * cplane + pt] = make_float2(end * acc.x, endi * acc.y);
  }
}

// ---------------------------------------------------------------------------
// PolarNufft
// ---------------------------------------------------------------------------

// Fine-grid size for at least m points: of the lengths below the smallest that
// holds m, when it exceeds the smallest even 2,3,5,7-smooth length by at most
// 1/8, else that smooth length.  The grid's size sets the kernel's aliasing
// error (about 1e-7 of the image's level), so it is a fixed rule and not
// whatever length has a fast plan.
static int grid_length(int m, bool even) {
  static const int kGrids[] = {512,  768,  1024, 1458, 1536, 2048, 2304, 2916,
                               3072, 4374, 4608, 5832, 6144, 8748, 11664};
  const int smooth = fft_next_smooth(m, even);
  for (int c : kGrids)
    if (c >= m) return c <= smooth + smooth / 8 ? c : smooth;
  return smooth;
}

PolarNufft::PolarNufft(const float* h_angles, int nproj, int npix, int nmodes)
    : P_(nproj), N_(npix), nm_(nmodes) {
  ArenaPause no_arena;  // cached plan, tables filled synchronously
  TC_REQUIRE(nproj >= 1 && npix >= 2 && nmodes >= 1, "NUFFT: bad geometry");
  // (a limit of the FP32 entry points; the lists would take more)
  TC_REQUIRE(nproj <= 2048, "NUFFT: too many projection angles");
  TC_REQUIRE(npix < 65536, "NUFFT: too many samples per ray");
  nf_ = grid_length(std::max(2 * nmodes, 2 * NUFFT_W), true);
  beta_ = (float)(2.30 * NUFFT_W);
  std::vector<double> hx(P_), hy(P_);
  const double sc = (double)nf_ / (double)(npix - 1);
  for (int p = 0; p < P_; ++p) {
    const double th = (double)h_angles[p];
    hx[p] = std::cos(th) * sc;
    hy[p] = std::sin(th) * sc;
  }
  ax_.alloc(sizeof(double) * P_);
  ay_.alloc(sizeof(double) * P_);
  TC_HIP(hipMemcpy(ax_.as<void>(), hx.data(), sizeof(double) * P_,
                   hipMemcpyHostToDevice));
  TC_HIP(hipMemcpy(ay_.as<void>(), hy.data(), sizeof(double) * P_,
                   hipMemcpyHostToDevice));
  // corr(k) = (-1)^k h / psi_hat(k) = (-1)^k 2 / (w int phi(z) cos(k z w h/2))
  std::vector<double> zq, wq;
  gauss_legendre(120, zq, wq);
  const double h = 2.0 * M_PI / nf_;
  const double beta = (double)beta_;
  std::vector<float> corr(nm_);
  for (int ki = 0; ki < nm_; ++ki) {
    const int k = ki - nm_ / 2;
    double integ = 0.0;
    for (size_t q = 0; q < zq.size(); ++q) {
      const double z = zq[q];
      const double phi = std::exp(beta * (std::sqrt(1.0 - z * z) - 1.0));
      integ += wq[q] * phi * std::cos(k * z * NUFFT_W * h / 2.0);
    }
    double c = 2.0 / (NUFFT_W * integ);
    if (k & 1) c = -c;
    corr[ki] = (float)c;
  }
  fft_prepare(nf_);
  corr_.alloc(sizeof(float) * nm_);
  TC_HIP(hipMemcpy(corr_.as<void>(), corr.data(), sizeof(float) * nm_,
                   hipMemcpyHostToDevice));
}

float2* PolarNufft::fine(int batch) {
  if (batch > fine_batch_) {
    fine_.alloc(sizeof(float2) * (size_t)batch * half_grid_size(nf_));
    fine_batch_ = batch;
  }
  return fine_.as<float2>();
}

SpreadArgs PolarNufft::spread_args() const {
  SpreadArgs a{};
  a.g.ax = ax_.as<double>();
  a.g.ay = ay_.as<double>();
  a.g.P = P_;
  a.g.cidx = N_ / 2;
  a.g.N = 2 * a.g.cidx + 1;  // both ends of an even ray (halved values)
  a.g.nf = nf_;
  a.g.ncols = nf_ / 2 + 1;
  a.g.ntx = (int)cdiv(a.g.ncols, SP_T);
  a.g.umax = a.g.cidx * ((double)nf_ / (N_ - 1)) + 1.0;
  lists_.fill(a.g);
  a.nh = nh();
  a.beta = beta_;
  return a;
}

// Spreading chunks picked by the autotuner, keyed by (device, angles, ray
// samples, fine grid, modes): later plans of the geometry, including those
// of concurrent batch workers (which do not tune), use the choice.
static std::mutex g_chunk_mu;
static std::map<std::tuple<int, int, int, int, int>, int> g_chunk_tuned;

static std::tuple<int, int, int, int, int> chunk_key(int P, int N, int nf,
                                                     int nm) {
  int dev = 0;
  TC_HIP(hipGetDevice(&dev));
  return std::make_tuple(dev, P, N, nf, nm);
}

// Slices per fine-grid batch: about 1 GB of fine grid, in whole groups of
// SP_SB slices (a spreading workgroup accumulates up to SP_SB slices; a
// partial group idles part of its matrix products and repeats the tile's
// point set-up for fewer slices), rounding up while that stays within
// 1.25 GB.
constexpr int SP_SB = 8;
static int fine_batch(int nf, int S) {
  const double per = 8.0 * (double)half_grid_size(nf), budget = 1.0e9;
  const int b0 = (int)std::max(1.0, std::floor(budget / per));
  int b = b0;
  const int up = (b0 + SP_SB - 1) / SP_SB * SP_SB;
  if (up * per <= 1.25 * budget)
    b = up;
  else if (b0 >= SP_SB)
    b = b0 / SP_SB * SP_SB;
  return std::max(1, std::min(S, b));
}

void PolarNufft::type1_real(const float2* c, float* out, int S, float scale,
                            hipStream_t stream) {
  TC_REQUIRE(S >= 1, "NUFFT: need at least one slice");
  const int B = fine_batch(nf_, S);
  float2* fg = fine(B);
  // slices a spreading workgroup takes: a point's weights and footprint serve
  // all of them, so as many as there are, up to 8 (64 accumulators a lane)
  auto group = [](int nb) { return nb <= 2 ? 2 : nb <= 4 ? 4 : SP_SB; };
  auto args = [&](int s0, int nb) {
    SpreadArgs a = spread_args();
    a.c = c + (long)s0 * P_ * nh();
    a.fine = fg;
    a.nsl = nb;
    return a;
  };
  // the fine grid of nb slices from the current work lists
  auto spread = [&](const SpreadArgs& a, int nb, float2* scratch) {
    const int sb = group(nb);
    const unsigned ng = cdiv(nb, sb);
    auto k = sb == 2 ? spread_kernel<2> : sb == 4 ? spread_kernel<4>
                                                  : spread_kernel<SP_SB>;
    hipLaunchKernelGGL(k, dim3((unsigned)lists_.nwork(), ng),
                       dim3(64 * SP_WAVES), 0, stream, a,
                       lists_.work(), scratch);
    TC_HIP(hipGetLastError());
    if (lists_.nfix()) {
      hipLaunchKernelGGL(spread_fixup_kernel,
                         dim3((unsigned)(lists_.nfix() + 3 * lists_.nheavy()),
                              ng, sb),
                         dim3(256), 0, stream, a, lists_.fix(),
                         lists_.nheavy(), scratch, sb);
      TC_HIP(hipGetLastError());
    }
  };
  auto scratch_bytes = [&](int nb) {
    const int sb = group(nb);
    return sizeof(float2) * (size_t)std::max(lists_.nslots(), 1) * cdiv(nb, sb) * sb *
           SP_T * SP_T;
  };
  if (!work_ready_) {
    lists_.make_segments(spread_args().g, NUFFT_W, stream);
    // Points per work item: TOMOCAM_HIP_SPREAD_CHUNK (>= 64), else the
    // autotuner's choice for this geometry, else (tuning allowed) the
    // fastest of the rule's choice and two others near it on this call's first
    // batch: best of two timed runs after a warm-up, the rule's choice kept
    // unless another is >= 5 % and >= 20 us faster (events and launches of
    // small grids scatter by some microseconds).  The chunk sets the order in which a
    // tile's points are summed, so the wide margin keeps near-ties (2048 is
    // within 0.7-1.3 % of 1024 on large grids) on the rule's choice and the
    // results the same from process to process.  Each work item writes its
    // own tile or slot, so a timing run only rewrites the fine grid.
    int chunk = 0;
    const char* e = std::getenv("TOMOCAM_HIP_SPREAD_CHUNK");
    if (e && std::atoi(e) >= 64) chunk = std::atoi(e);
    const auto key = chunk_key(P_, N_, nf_, nm_);
    if (!chunk) {
      std::lock_guard<std::mutex> lk(g_chunk_mu);
      auto it = g_chunk_tuned.find(key);
      if (it != g_chunk_tuned.end()) chunk = it->second;
    }
    if (!chunk && autotune_enabled()) {
      constexpr float kMargin = 0.05f, kMarginMs = 0.02f;
      const int nb = std::min(B, S);
      const int rule = lists_.rule_chunk();
      std::vector<int> cands{rule};
      if (rule < 512)
        cands.insert(cands.end(), {384 - rule, 512});  // 128 and 256, 512
      else
        for (int k : {512, 1024, 2048})
          if (k != rule) cands.push_back(k);
      hipEvent_t e0, e1;
      TC_HIP(hipEventCreate(&e0));
      TC_HIP(hipEventCreate(&e1));
      float best_ms = 0.f;
      try {
        for (int k : cands) {
          lists_.make_work(k);
          DevBuf scr(scratch_bytes(nb));
          float ms = 0.f;
          for (int rep = 0; rep < 3; ++rep) {
            TC_HIP(hipEventRecord(e0, stream));
            spread(args(0, nb), nb, scr.as<float2>());
            TC_HIP(hipEventRecord(e1, stream));
            TC_HIP(hipEventSynchronize(e1));
            float t = 0.f;
            TC_HIP(hipEventElapsedTime(&t, e0, e1));
            if (rep == 1 || (rep > 1 && t < ms)) ms = t;
          }
          if (tune_log())
            std::fprintf(stderr,
                         "[tomocam] spread tune %d angles x %d, grid %d, %d "
                         "slices: chunk %d: %.3f ms\n", P_, N_, nf_, nb, k,
                         (double)ms);
          if (chunk == 0 ||
              ms < std::min((1.0f - kMargin) * best_ms, best_ms - kMarginMs)) {
            chunk = k;
            best_ms = ms;
          }
        }
      } catch (...) {
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        throw;
      }
      (void)hipEventDestroy(e0);
      (void)hipEventDestroy(e1);
      std::lock_guard<std::mutex> lk(g_chunk_mu);
      g_chunk_tuned[key] = chunk;
    }
    if (!chunk) chunk = lists_.rule_chunk();
    if (chunk != lists_.chunk()) lists_.make_work(chunk);
    work_ready_ = true;
  }
  DevBuf scratch(scratch_bytes(B));
  for (int s0 = 0; s0 < S; s0 += B) {
    const int nb = std::min(B, S - s0);
    const SpreadArgs a = args(s0, nb);
    spread(a, nb, scratch.as<float2>());
    // columns to the mode rows, then real rows
    columns(nb, +1, stream);
    RealRowsArgs r = real_rows(nb);
    r.real_out = out + (long)s0 * nm_ * nm_;
    r.scale = scale;
    fft_real_rows(r, false, stream);
  }
  // the scratch slots are released on return: to the thread's arena
  // (reused in stream order) or by hipFree, which waits for the device
}

void PolarNufft::type2_real(const float* f, float2* c, int S,
                            hipStream_t stream) {
  TC_REQUIRE(S >= 1, "NUFFT: need at least one slice");
  const int B = fine_batch(nf_, S);
  float2* fg = fine(B);
  for (int s0 = 0; s0 < S; s0 += B) {
    const int nb = std::min(B, S - s0);
    RealRowsArgs r = real_rows(nb);
    r.real_in = f + (long)s0 * nm_ * nm_;
    fft_real_rows(r, true, stream);
    columns(nb, -1, stream);
    InterpArgs a;
    a.fine = fg;
    a.c = c + (long)s0 * P_ * nh();
    a.ax = ax_.as<double>();
    a.ay = ay_.as<double>();
    a.P = P_;
    a.N = N_;
    a.nh = nh();
    a.nf = nf_;
    a.nsl = nb;
    a.beta = beta_;
    hipLaunchKernelGGL(interp_kernel, dim3(cdiv(8L * P_ * a.nh, 256)),
                       dim3(256), 0, stream, a);
    TC_HIP(hipGetLastError());
  }
}

RealRowsArgs PolarNufft::real_rows(int nsl) const {
  RealRowsArgs r;
  r.half = fine_.as<float2>();
  r.corr = corr_.as<float>();
  r.L = nf_;
  r.nm = nm_;
  r.nsl = nsl;
  return r;
}

// Column transforms of the half grid in place; of the rows only those of the
// modes are non-zero on input (dir -1) or wanted on output (dir +1).
void PolarNufft::columns(int nsl, int dir, hipStream_t stream) {
  LineFFTArgs a;
  a.in = a.out = fine_.as<float2>();
  a.L = nf_;
  a.nbatch = nsl;
  a.lines_per_batch = nf_ / 2 + 1;
  a.bstride = half_grid_size(nf_);
  a.lgroup = HG_B;
  a.lstride = (long)nf_ * HG_B;
  a.estride = HG_B;
  a.colmajor = true;
  const int lo = (nm_ + 1) / 2, hi = nm_ / 2;
  a.nin = dir < 0 ? lo : nf_;
  a.nin_hi = dir < 0 ? hi : 0;
  a.nout = dir < 0 ? nf_ : lo;
  a.nout_hi = dir < 0 ? 0 : hi;
  fft_lines(a, dir, stream);
}

// ---------------------------------------------------------------------------
// Bluestein ray DFT
// ---------------------------------------------------------------------------

RayDft::RayDft(int N, int sign) : N_(N) {
  ArenaPause no_arena;  // cached plan, tables filled synchronously
  TC_REQUIRE(N >= 1, "ray DFT: N must be >= 1");
  direct_ = fft_lines_ct_has(N);
  if (direct_) fft_prepare(N);
  // The chirp-z length.  Backward a planned FFT length where there is one (the
  // planned kernel runs forward transform, multiply and inverse in registers).
  // Forward the rule of the fine grids, whose lengths have a plan at about half of
  // the widths: another length rounds P x differently, which residuals P x - y
  // amplify (es_kernel above).
  if (sign < 0) {
    const int c = fft_lines_ct_length(2 * N - 1);
    L_ = c > 0 ? c : fft_next_smooth(2 * N - 1, false);
  } else {
    L_ = grid_length(2 * N - 1, false);
  }
  const int c = N / 2;
  const long twoN = 2L * N;
  std::vector<float2> ch(N), b(L_, make_float2(0.f, 0.f));
  for (int z = 0; z < N; ++z) {
    const long m = z - c;
    const double ph = sign * M_PI * (double)((m * m) % twoN) / N;
    ch[z] = make_float2((float)std::cos(ph), (float)std::sin(ph));
  }
  for (long m = -(N - 1); m <= N - 1; ++m) {
    const double ph = -sign * M_PI * (double)((m * m) % twoN) / N;
    const long idx = m >= 0 ? m : L_ + m;
    b[idx] = make_float2((float)(std::cos(ph) / L_), (float)(std::sin(ph) / L_));
  }
  chirp_.alloc(sizeof(float2) * N);
  bhat_.alloc(sizeof(float2) * L_);
  TC_HIP(hipMemcpy(chirp_.as<void>(), ch.data(), sizeof(float2) * N,
                   hipMemcpyHostToDevice));
  TC_HIP(hipMemcpy(bhat_.as<void>(), b.data(), sizeof(float2) * L_,
                   hipMemcpyHostToDevice));
  LineFFTArgs a;
  a.in = bhat_.as<float2>();
  a.out = bhat_.as<float2>();
  a.L = L_;
  a.lines_per_batch = 1;
  a.nbatch = 1;
  a.lstride = L_;
  a.bstride = L_;
  a.nin = L_;
  a.nout = L_;
  fft_lines(a, -1, nullptr);
  TC_HIP(hipDeviceSynchronize());
}

void RayDft::to_half(const float* in, float2* out, int nsl, int P, bool ramp,
                     float scale, hipStream_t stream) {
  RayArgs a;
  a.real_in = in;
  a.half_out = out;
  a.nsl = nsl;
  a.P = P;
  a.ramp = ramp;
  a.scale = scale;
  run(a, true, stream);
}

void RayDft::to_real(const float2* in, float* out, int nsl, int P, float scale,
                     hipStream_t stream) {
  RayArgs a;
  a.half_in = in;
  a.real_out = out;
  a.nsl = nsl;
  a.P = P;
  a.scale = scale;
  run(a, false, stream);
}

void RayDft::run(RayArgs a, bool to_half, hipStream_t stream) {
  a.chirp = chirp_.as<float2>();
  a.bhat = bhat_.as<float2>();
  a.N = N_;
  a.nh = N_ / 2 + 1;
  a.L = L_;
  if (direct_ && fft_ct_enabled()) a.L = N_;
  fft_rays(a, to_half, stream);
}

// ---------------------------------------------------------------------------
// plan caches
// ---------------------------------------------------------------------------

// A PolarNufft keeps scratch (the fine grid) between calls, so threads that
// run concurrently use plans of their own: the cache key holds a plan slot,
// taken by each thread on its first plan request from a pool (lowest free
// number) and given back when the thread ends.  Threads that follow one
// another, such as the batch workers of successive calls, reuse the slots
// and with them the cached plans.
static std::mutex g_slot_mu;
static std::vector<char> g_slot_used;

struct PlanSlot {
  int id = -1;
  ~PlanSlot() {
    if (id >= 0) {
      std::lock_guard<std::mutex> lk(g_slot_mu);
      g_slot_used[id] = 0;
    }
  }
};
static thread_local PlanSlot t_slot;

static int plan_slot() {
  if (t_slot.id < 0) {
    std::lock_guard<std::mutex> lk(g_slot_mu);
    int i = 0;
    while (i < (int)g_slot_used.size() && g_slot_used[i]) ++i;
    if (i == (int)g_slot_used.size()) g_slot_used.push_back(0);
    g_slot_used[i] = 1;
    t_slot.id = i;
  }
  return t_slot.id;
}

PolarNufft& nufft_plan(const float* h_angles, int nproj, int npix,
                       int nmodes) {
  static std::mutex mu;
  using Key = std::tuple<int, int, int, int, int, std::vector<float>>;
  static std::map<Key, std::unique_ptr<PolarNufft>> cache;
  int dev = 0;
  TC_HIP(hipGetDevice(&dev));
  std::vector<float> ang(h_angles, h_angles + nproj);
  const int slot = plan_slot();
  Key key(slot, dev, nproj, npix, nmodes, ang);
  std::lock_guard<std::mutex> lk(mu);
  auto it = cache.find(key);
  if (it == cache.end()) {
    // at most 16 plans per slot: drop this slot's (only this thread uses
    // them, and it holds none while it asks for a plan)
    int mine = 0;
    for (auto& kv : cache) mine += std::get<0>(kv.first) == slot;
    if (mine >= 16)
      for (auto i = cache.begin(); i != cache.end();)
        i = std::get<0>(i->first) == slot ? cache.erase(i) : std::next(i);
    it = cache
             .emplace(key, std::make_unique<PolarNufft>(h_angles, nproj, npix,
                                                        nmodes))
             .first;
  }
  return *it->second;
}

RayDft& ray_dft_plan(int N, int sign) {
  static std::mutex mu;
  static std::map<std::tuple<int, int, int>, std::unique_ptr<RayDft>> cache;
  int dev = 0;
  TC_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lk(mu);
  auto key = std::make_tuple(dev, N, sign);
  auto it = cache.find(key);
  if (it == cache.end())
    it = cache.emplace(key, std::make_unique<RayDft>(N, sign)).first;
  return *it->second;
}

// ---------------------------------------------------------------------------
// projectors
// ---------------------------------------------------------------------------

void project(const float* img, float* sino, int S, int N, const float* h_angles,
             int P, hipStream_t stream) {
  TC_REQUIRE(S >= 1 && N >= 2 && P >= 1, "project: bad shape");
  PolarNufft& nu = nufft_plan(h_angles, P, N, N);
  RayDft& rd = ray_dft_plan(N, +1);
  DevBuf c(sizeof(float2) * (size_t)S * P * nu.nh());
  nu.type2_real(img, c.as<float2>(), S, stream);
  rd.to_real(c.as<float2>(), sino, S, P, 1.0f / ((float)N * (float)N), stream);
}

void backproject(const float* sino, float* img, int S, int P, int N,
                 const float* h_angles, bool fbp, hipStream_t stream) {
  TC_REQUIRE(S >= 1 && N >= 2 && P >= 1, "backproject: bad shape");
  PolarNufft& nu = nufft_plan(h_angles, P, N, N);
  RayDft& rd = ray_dft_plan(N, -1);
  DevBuf c(sizeof(float2) * (size_t)S * P * nu.nh());
  rd.to_half(sino, c.as<float2>(), S, P, fbp, 1.0f, stream);
  nu.type1_real(c.as<float2>(), img, S, 1.0f / ((float)N * (float)N), stream);
}

// unit samples, the end of an even ray halved (RayArgs)
__global__ void fill_ones_kernel(float2* c, long n, int nh, int N) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) c[i] = make_float2(2 * (int)(i % nh) == N ? 0.5f : 1.f, 0.f);
}

void polar_psf(const float* h_angles, int P, int n, float* d_psf,
               hipStream_t stream) {
  TC_REQUIRE(P >= 1 && n >= 2, "PSF: bad geometry");
  PolarNufft& nu = nufft_plan(h_angles, P, n, 2 * n - 1);
  const long tot = (long)P * nu.nh();
  DevBuf ones(sizeof(float2) * (size_t)tot);
  hipLaunchKernelGGL(fill_ones_kernel, dim3(cdiv(tot, 256)), dim3(256), 0,
                     stream, ones.as<float2>(), tot, nu.nh(), n);
  TC_HIP(hipGetLastError());
  nu.type1_real(ones.as<float2>(), d_psf, 1, 1.0f, stream);
  TC_HIP(hipStreamSynchronize(stream));
}

}  // namespace tc
