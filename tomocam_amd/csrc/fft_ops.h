// Host-callable FFT operations built on the LDS Stockham kernels.
#pragma once

#include "tc_common.h"

namespace tc {

struct LineFFTArgs {
  const float2* in = nullptr;
  float2* out = nullptr;  // may equal `in`
  int L = 0;               // transform length (2,3,5,7-smooth)
  int lines_per_batch = 0;
  int nbatch = 1;
  long bstride = 0;   // complex elements between batches
  long lstride = 0;   // complex elements between groups of lines
  int lgroup = 1;     // adjacent lines (element distance 1) in a group
  long estride = 1;   // complex elements between elements of a line
  int nin = 0;        // leading input elements read (rest treated as zero)
  int nout = 0;       // leading output elements written
  int nin_hi = 0;     // trailing input elements read as well
  int nout_hi = 0;    // trailing output elements written as well
  bool colmajor = false;  // lines adjacent in memory (column transforms)
  float scale = 1.0f;
};

// dir = -1: exp(-2 pi i k n / L) (forward); +1: exp(+2 pi i k n / L); both
// unnormalised (times `scale`).  Lengths with a compile-time line plan run
// on it (fft_lines_ct.hip) unless TOMOCAM_HIP_CT_LINES=0; others on the
// runtime-plan kernel.
void fft_lines(const LineFFTArgs& a, int dir, hipStream_t stream);

// Storage of the non-redundant half (columns 0 .. L/2) of an L x L Hermitian
// grid: blocks of HG_B columns, each block row by row.  A column's elements
// are HG_B apart and two adjacent rows share 2 HG_B adjacent elements, so
// neither the column pass (8 useful bytes in each line it touches, row by row)
// nor the row pass (the same, column by column) pays for the other; the
// spreading's regions of 4 x 16 cells are whole cache lines.  Against whole
// rows (columns / interpolation / rows to image, us): 593 / - / 145 -> 270 / -
// / 154 at 8 x 2048^2 on 4374^2, 95 / 117 / - -> 55 / 91 / - at 8 x 1024^2 and
// 720 angles on 2048^2.  Blocks of 2: columns 45, but interpolation 1.5 times as
// long; of 8: columns 85.
constexpr int HG_B = 4;
__host__ __device__ __forceinline__ long half_grid_size(int L) {
  return (long)L * ((L / 2 + HG_B) / HG_B * HG_B);
}
// element of a slice; below 2^31 for every L whose lines fit in LDS
__device__ __forceinline__ unsigned half_at(int L, int row, int col) {
  return (unsigned)(((col / HG_B) * L + row) * HG_B + col % HG_B);
}

// Rows of nm real modes <-> the half of an L x L Hermitian grid.  Mode index k
// stands for k - floor(nm/2); row k of slice s is grid row (k - floor(nm/2))
// mod L.
//   r2c: half = forward row transforms of real_in, each value times
//        corr[row] corr[column]; only the nm mode rows are written;
//   c2r: real_out = scale corr corr times the inverse (exp(+i), unnormalised)
//        transforms of the mode rows.
struct RealRowsArgs {
  const float* real_in = nullptr;  // [nsl][nm][nm]
  float* real_out = nullptr;       // [nsl][nm][nm]
  float2* half = nullptr;          // [nsl][half_grid_size(L)]
  const float* corr = nullptr;     // [nm]
  int L = 0, nm = 0, nsl = 0;
  float scale = 1.0f;
};
void fft_real_rows(const RealRowsArgs& a, bool r2c, hipStream_t stream);

// Centred DFTs V[j] = sum_z a[z] exp(sign 2 pi i (j - c)(z - c) / N),
// c = floor(N/2), between nsl x P real rays of N samples and their half
// spectra: nh = c + 1 values, V at j - c = 0 .. c.  The other half is its
// conjugate.  For even N the last value stands for both j - c = -c (the DFT's
// own sample) and +c, and is stored halved, so that the samples
// -c .. c weighted alike are the exact DFT.
//   to_half: half_out = scale (|j - c| / N if ramp) V of real_in;
//   else:    real_out = scale V of half_in.
struct RayArgs {
  const float* real_in = nullptr;    // [nsl][P][N]
  float* real_out = nullptr;         // [nsl][P][N]
  const float2* half_in = nullptr;   // [nsl][P][nh]
  float2* half_out = nullptr;        // [nsl][P][nh]
  const float2* chirp = nullptr;     // [N]
  const float2* bhat = nullptr;      // [L]
  int N = 0, nh = 0, P = 0, nsl = 0, L = 0;
  bool ramp = false;
  float scale = 1.0f;
};

void fft_rays(const RayArgs& a, bool to_half, hipStream_t stream);

// Sample t (centred, -c .. c) of ray a plus i times ray b (b may be null).
__device__ __forceinline__ float2 ray_pair_sample(const float2* pa,
                                                  const float2* pb, int t,
                                                  int N) {
  const int m = t < 0 ? -t : t;
  float2 a = pa[m], b = pb ? pb[m] : make_float2(0.f, 0.f);
  if (t < 0) {
    a.y = -a.y;
    b.y = -b.y;
  }
  if (2 * m == N) {  // the halves of +c and -c, added
    a = make_float2(2.f * a.x, 0.f);
    b = make_float2(2.f * b.x, 0.f);
  }
  return make_float2(a.x - b.y, a.y + b.x);
}

// With the ramp: a level near the ray's mean, taken off before the transform
// (the DFT of a constant is N at j = c, where the ramp is 0, and 0 elsewhere).
// The transform's rounding is relative to what is left, which for projections
// of an object is a fraction of the whole, and the ramp would amplify it (FBP
// of 16 x 333^2 against 64 bits: 2.6e-6 without, 1.9e-6 with).  The mean of the
// middle four of eight samples: a hot pixel at one of them would raise the mean
// of all, and with it the whole ray, by an eighth of its value (FBP of 1531
// samples with a pixel 10^4 times the rest: 1.0e-6 with the mean, 3.3e-7).
__device__ __forceinline__ float ray_level(const RayArgs& a, const float* ray) {
  if (!a.ramp) return 0.f;
  float v[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) v[k] = ray[(long)(2 * k + 1) * a.N / 16];
  auto order = [&](int i, int j) {
    const float lo = fminf(v[i], v[j]), hi = fmaxf(v[i], v[j]);
    v[i] = lo;
    v[j] = hi;
  };
#pragma unroll
  for (int h = 0; h < 8; h += 4) {  // either half in ascending order
    order(h, h + 1);
    order(h + 2, h + 3);
    order(h, h + 2);
    order(h + 1, h + 3);
    order(h + 1, h + 2);
  }
  // halves against each other: the four lowest and the four highest, each a
  // bitonic sequence, of which the upper and the lower two are taken
  float lo[4], hi[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    lo[i] = fminf(v[i], v[7 - i]);
    hi[i] = fmaxf(v[i], v[7 - i]);
  }
  return 0.25f * ((fmaxf(lo[0], lo[2]) + fmaxf(lo[1], lo[3])) +
                  (fminf(hi[0], hi[2]) + fminf(hi[1], hi[3])));
}

// Value m of ray pair `pair` from z = V_a + i V_b at +m (zp; for m = N/2 the
// value at -m) and at -m (zn).
__device__ __forceinline__ void ray_store_pair(const RayArgs& a, long pair,
                                               float2 zp, float2 zn, int m) {
  const int npair = (a.P + 1) / 2;
  const long s = pair / npair;
  const int p = 2 * (int)(pair - s * npair);
  float f = 0.5f * a.scale;
  if (a.ramp) f *= (float)m / (float)a.N;
  if (2 * m == a.N) f *= 0.5f;
  float2* o = a.half_out + (s * a.P + p) * a.nh + m;
  o[0] = make_float2(f * (zp.x + zn.x), f * (zp.y - zn.y));
  if (p + 1 < a.P) o[a.nh] = make_float2(f * (zp.y + zn.y), f * (zn.x - zp.x));
}

// The compile-time line plans: whether L has one, the smallest planned
// length >= n (0: none), and the transforms (false: no plan for the length).
bool fft_lines_ct_has(int L);
int fft_lines_ct_length(int n);
// Lays out the twiddle tables of length L, so that no later call does (a first
// transform may run under stream capture).
void fft_prepare(int L);
bool fft_lines_ct(const LineFFTArgs& a, int dir, hipStream_t stream);
bool fft_real_rows_ct(const RealRowsArgs& a, bool r2c, hipStream_t stream);
bool fft_rays_ct(const RayArgs& a, bool to_half, hipStream_t stream);
// False with TOMOCAM_HIP_CT_LINES=0: the runtime-plan kernels only.
bool fft_ct_enabled();

// In-place unnormalised 2D transform of `nbatch` complex [rows][cols] arrays.
void fft2d(float2* data, int nbatch, int rows, int cols, long row_pitch,
           long slice_pitch, int dir, hipStream_t stream);

// The same on contiguous [n][n] arrays when only the columns [0, lo) and
// [n - hi, n) matter: rows_first transforms every row, then only those
// columns (the other columns of the result are left unfinished); otherwise
// those columns are transformed first (the others must be zero on input)
// and then every row.
void fft2d_pruned(float2* data, int nbatch, int n, int lo, int hi, int dir,
                  bool rows_first, hipStream_t stream);

}  // namespace tc
