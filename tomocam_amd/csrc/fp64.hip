// FP64 forms of the hot path (declarations and scope in fp64.h).
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <functional>
#include <list>
#include <map>
#include <memory>
#include <mutex>
#include <tuple>
#include <utility>
#include <vector>

#include "driver.h"
#include "fft_ct.h"
#include "fp64.h"

namespace tc {
namespace f64 {

// ---------------------------------------------------------------------------
// complex helpers
// ---------------------------------------------------------------------------

__device__ __forceinline__ double2 zadd(double2 a, double2 b) {
  return make_double2(a.x + b.x, a.y + b.y);
}
__device__ __forceinline__ double2 zsub(double2 a, double2 b) {
  return make_double2(a.x - b.x, a.y - b.y);
}
__device__ __forceinline__ double2 zmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
// a * conj(b)
__device__ __forceinline__ double2 zmulc(double2 a, double2 b) {
  return make_double2(a.x * b.x + a.y * b.y, a.y * b.x - a.x * b.y);
}

// ---------------------------------------------------------------------------
// FFT: runtime-planned Stockham transform of lines held in LDS
// ---------------------------------------------------------------------------

constexpr int kMaxStages = 24;

struct Plan {
  int L;
  int nst;
  int radix[kMaxStages];
  const double2* tw;  // tw[m] = exp(-2 pi i m / L)
};

static std::vector<int> factor(int L) {
  TC_REQUIRE(L >= 1 && L <= kMaxFFT,
             "FP64 FFT length " + std::to_string(L) + " outside [1, " +
                 std::to_string(kMaxFFT) + "]");
  std::vector<int> r;
  int m = L;
  while (m % 4 == 0) {
    r.push_back(4);
    m /= 4;
  }
  for (int p : {2, 3, 5, 7})
    while (m % p == 0) {
      r.push_back(p);
      m /= p;
    }
  TC_REQUIRE(m == 1, "FP64 FFT length " + std::to_string(L) +
                         " is not a product of 2, 3, 5, 7");
  TC_REQUIRE((int)r.size() <= kMaxStages, "FP64 FFT length too large");
  return r;
}

static int smooth_at_least(int n) {
  for (int m = std::max(n, 1);; ++m) {
    int r = m;
    for (int p : {2, 3, 5, 7})
      while (r % p == 0) r /= p;
    if (r == 1) return m;
  }
}

class Length {
 public:
  explicit Length(int L) {
    ArenaPause no_arena;  // process-lifetime table, filled synchronously
    std::vector<int> r = factor(L);
    p_.L = L;
    p_.nst = (int)r.size();
    for (int i = 0; i < p_.nst; ++i) p_.radix[i] = r[i];
    std::vector<double2> h(L);
    for (int m = 0; m < L; ++m) {
      const double a = -2.0 * M_PI * (double)m / (double)L;
      h[m] = make_double2(std::cos(a), std::sin(a));
    }
    tw_.alloc(sizeof(double2) * L);
    TC_HIP(hipMemcpy(tw_.as<void>(), h.data(), sizeof(double2) * L,
                     hipMemcpyHostToDevice));
    p_.tw = tw_.as<double2>();
  }
  const Plan& plan() const { return p_; }

 private:
  Plan p_;
  DevBuf tw_;
};

// exp(-2 pi i m / N), m < N, for any N (the ray DFT's roots)
class Roots {
 public:
  explicit Roots(int N) {
    ArenaPause no_arena;  // process-lifetime table, filled synchronously
    std::vector<double2> h(N);
    for (int m = 0; m < N; ++m) {
      const double a = -2.0 * M_PI * (double)m / (double)N;
      h[m] = make_double2(std::cos(a), std::sin(a));
    }
    t_.alloc(sizeof(double2) * N);
    TC_HIP(hipMemcpy(t_.as<void>(), h.data(), sizeof(double2) * N,
                     hipMemcpyHostToDevice));
  }
  const double2* table() const { return t_.as<double2>(); }

 private:
  DevBuf t_;
};

static const double2* roots(int N) {
  static std::mutex mu;
  static std::map<std::pair<int, int>, std::unique_ptr<Roots>> cache;
  int dev = 0;
  TC_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lk(mu);
  auto key = std::make_pair(dev, N);
  auto it = cache.find(key);
  if (it == cache.end())
    it = cache.emplace(key, std::make_unique<Roots>(N)).first;
  return it->second->table();
}

static const Length& length(int L) {
  static std::mutex mu;
  static std::map<std::pair<int, int>, std::unique_ptr<Length>> cache;
  int dev = 0;
  TC_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lk(mu);
  auto key = std::make_pair(dev, L);
  auto it = cache.find(key);
  if (it == cache.end())
    it = cache.emplace(key, std::make_unique<Length>(L)).first;
  return *it->second;
}

// radix-R DFT of a[0..R) in place, the roots as constants
template <int R, int DIR>
__device__ __forceinline__ void dft_small(double2* a) {
  if constexpr (R == 2) {
    const double2 t = a[1];
    a[1] = zsub(a[0], t);
    a[0] = zadd(a[0], t);
  } else if constexpr (R == 4) {
    const double2 t0 = zadd(a[0], a[2]), t1 = zsub(a[0], a[2]);
    const double2 t2 = zadd(a[1], a[3]), d = zsub(a[1], a[3]);
    // d * (DIR i)
    const double2 t3 = DIR < 0 ? make_double2(d.y, -d.x)
                               : make_double2(-d.y, d.x);
    a[0] = zadd(t0, t2);
    a[2] = zsub(t0, t2);
    a[1] = zadd(t1, t3);
    a[3] = zsub(t1, t3);
  } else {
    double2 out[R];
#pragma unroll
    for (int k = 0; k < R; ++k) {
      double2 acc = a[0];
#pragma unroll
      for (int r = 1; r < R; ++r) {
        const double2 w = make_double2(ct::cx_cos2pi(r * k, R),
                                       DIR * ct::cx_sin2pi(r * k, R));
        acc = zadd(acc, zmul(a[r], w));
      }
      out[k] = acc;
    }
#pragma unroll
    for (int k = 0; k < R; ++k) a[k] = out[k];
  }
}

// One Stockham stage of radix R on the LDS line: each thread holds up to 4
// butterflies (read, twiddle, DFT), then writes them after a barrier.
template <int R, int DIR>
__device__ __forceinline__ void lds_stage(double2* buf, int L, int Ns,
                                          const double2* __restrict__ tw) {
  const int nb = L / R;
  const int nthr = blockDim.x;
  double2 v[4][R];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int j = threadIdx.x + q * nthr;
    if (j < nb) {
      const int k = j % Ns;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        double2 x = buf[j + r * nb];
        if (r > 0 && Ns > 1) {
          const double2 w = tw[(long)r * k * (L / (Ns * R))];
          x = DIR < 0 ? zmul(x, w) : zmulc(x, w);
        }
        v[q][r] = x;
      }
      dft_small<R, DIR>(v[q]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int j = threadIdx.x + q * nthr;
    if (j < nb) {
      const int k = j % Ns;
      const int o = (j - k) * R + k;
#pragma unroll
      for (int r = 0; r < R; ++r) buf[o + r * Ns] = v[q][r];
    }
  }
  __syncthreads();
}

// Lines l < nlines: element e of line l is at
//   (l / lpb) * bstride + (l % lpb) * lstride + e * estride.
// The first nin elements are read (the rest are zero), the first nout are
// written, times `scale`.  One workgroup per line.
// Lines whose number within the batch is in [skip0, skip1) are left alone.
struct LineArgs {
  const double2* in;
  double2* out;
  long nlines;
  long lpb, bstride, lstride, estride;
  int nin, nout;
  double scale;
  long skip0, skip1;
};

template <int DIR>
__global__ void __launch_bounds__(1024) lines_kernel(LineArgs a, Plan P) {
  extern __shared__ double2 buf[];
  const long l = blockIdx.x;
  const long lb = l % a.lpb;
  if (l >= a.nlines || (lb >= a.skip0 && lb < a.skip1)) return;
  const long base = (l / a.lpb) * a.bstride + lb * a.lstride;
  const int L = P.L;
  const int nthr = blockDim.x;
  for (int e = threadIdx.x; e < L; e += nthr)
    buf[e] = e < a.nin ? a.in[base + e * a.estride] : make_double2(0.0, 0.0);
  __syncthreads();
  int Ns = 1;
  for (int s = 0; s < P.nst; ++s) {
    const int R = P.radix[s];
    switch (R) {
      case 2: lds_stage<2, DIR>(buf, L, Ns, P.tw); break;
      case 3: lds_stage<3, DIR>(buf, L, Ns, P.tw); break;
      case 4: lds_stage<4, DIR>(buf, L, Ns, P.tw); break;
      case 5: lds_stage<5, DIR>(buf, L, Ns, P.tw); break;
      default: lds_stage<7, DIR>(buf, L, Ns, P.tw); break;
    }
    Ns *= R;
  }
  for (int e = threadIdx.x; e < a.nout; e += nthr) {
    const double2 x = buf[e];
    a.out[base + e * a.estride] = make_double2(x.x * a.scale, x.y * a.scale);
  }
}

// threads per line: one per radix-4 butterfly, up to 1024 (every thread holds at
// most 4 butterflies of a stage: L <= 8192)
static int line_threads(int L) {
  return std::min(1024, std::max(64, (L / 4 + 63) / 64 * 64));
}

static void run_lines(const LineArgs& a, int L, int dir, hipStream_t s) {
  if (a.nlines <= 0) return;
  const Plan& P = length(L).plan();
  const size_t smem = sizeof(double2) * (size_t)L;
  const int nthr = line_threads(L);
  TC_REQUIRE(a.nlines < (1L << 31), "FP64 FFT: too many lines");
  auto launch = [&](auto k) {
    if (smem > 64 * 1024)
      TC_HIP(hipFuncSetAttribute((const void*)k,
                                 hipFuncAttributeMaxDynamicSharedMemorySize,
                                 (int)smem));
    hipLaunchKernelGGL(k, dim3((unsigned)a.nlines), dim3(nthr), smem, s, a,
                       P);
  };
  if (dir < 0)
    launch(lines_kernel<-1>);
  else
    launch(lines_kernel<1>);
  TC_HIP(hipGetLastError());
}

// in-place unnormalised 2D transform of nbatch [rows][cols] arrays; the rows
// [skip, rows - keep) are zero on input if `zero_rows`, the columns
// [skip, cols - keep) are not wanted on output if `drop_cols`
static void fft2(double2* d, int nbatch, int rows, int cols, int dir,
                 hipStream_t s, long skip = 0, long keep = 0,
                 bool zero_rows = false, bool drop_cols = false) {
  LineArgs a{d, d, (long)nbatch * rows, rows, (long)rows * cols, cols, 1,
             cols, cols, 1.0, zero_rows ? skip : 0,
             zero_rows ? rows - keep : 0};
  run_lines(a, cols, dir, s);
  LineArgs b{d, d, (long)nbatch * cols, cols, (long)rows * cols, 1, cols,
             rows, rows, 1.0, drop_cols ? skip : 0,
             drop_cols ? cols - keep : 0};
  run_lines(b, rows, dir, s);
}

// ---------------------------------------------------------------------------
// small vector kernels
// ---------------------------------------------------------------------------

__global__ void zero_kernel(double2* p, long n) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = make_double2(0.0, 0.0);
}
static void zero(double2* p, long n, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(zero_kernel, dim3(cdiv(n, 256)), dim3(256), 0, s, p, n);
  TC_HIP(hipGetLastError());
}

// out = alpha a + beta b (b may be null: out = alpha a)
__global__ void axpby_kernel(const double* a, const double* b, double* out,
                             long n, double alpha, double beta) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = b ? alpha * a[i] + beta * b[i] : alpha * a[i];
}
static void axpby(const double* a, const double* b, double* out, long n,
                  double alpha, double beta, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(axpby_kernel, dim3(cdiv(n, 256)), dim3(256), 0, s, a, b,
                     out, n, alpha, beta);
  TC_HIP(hipGetLastError());
}

__global__ void fill_kernel(double* p, long n, double v) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

constexpr int kRedBlocks = 512;

__global__ void __launch_bounds__(256)
dot_kernel(const double* a, const double* b, long n, double* part) {
  __shared__ double red[256];
  double acc = 0.0;
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n;
       i += (long)gridDim.x * 256)
    acc += a[i] * b[i];
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// sum of part[0..n) in a fixed order into part[n]
__global__ void sum_kernel(double* part, int n) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    double t = 0.0;
    for (int i = 0; i < n; ++i) t += part[i];
    part[n] = t;
  }
}

static double reduce_host(double* part, int n, hipStream_t s) {
  hipLaunchKernelGGL(sum_kernel, dim3(1), dim3(64), 0, s, part, n);
  TC_HIP(hipGetLastError());
  double h = 0.0;
  TC_HIP(hipMemcpyAsync(&h, part + n, sizeof(double), hipMemcpyDeviceToHost,
                        s));
  TC_HIP(hipStreamSynchronize(s));
  return h;
}

double dot(const double* a, const double* b, long n, hipStream_t s) {
  DevBuf part(sizeof(double) * (kRedBlocks + 1));
  hipLaunchKernelGGL(dot_kernel, dim3(kRedBlocks), dim3(256), 0, s, a, b, n,
                     part.as<double>());
  TC_HIP(hipGetLastError());
  return reduce_host(part.as<double>(), kRedBlocks, s);
}

__global__ void __launch_bounds__(256)
max_kernel(const double* a, long n, double* part) {
  __shared__ double red[256];
  double m = -1.0e300;
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n;
       i += (long)gridDim.x * 256)
    m = fmax(m, a[i]);
  red[threadIdx.x] = m;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o)
      red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + o]);
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

static void minmax(const double* a, long n, double* mx, double* mn,
                   hipStream_t s) {
  DevBuf part(sizeof(double) * 2 * kRedBlocks);
  DevBuf neg(sizeof(double) * n);
  hipLaunchKernelGGL(max_kernel, dim3(kRedBlocks), dim3(256), 0, s, a, n,
                     part.as<double>());
  axpby(a, nullptr, neg.as<double>(), n, -1.0, 0.0, s);
  hipLaunchKernelGGL(max_kernel, dim3(kRedBlocks), dim3(256), 0, s,
                     neg.as<double>(), n, part.as<double>() + kRedBlocks);
  TC_HIP(hipGetLastError());
  std::vector<double> h(2 * kRedBlocks);
  TC_HIP(hipMemcpyAsync(h.data(), part.as<void>(),
                        sizeof(double) * 2 * kRedBlocks,
                        hipMemcpyDeviceToHost, s));
  TC_HIP(hipStreamSynchronize(s));
  double M = -1.0e300, m = -1.0e300;
  for (int i = 0; i < kRedBlocks; ++i) {
    M = std::max(M, h[i]);
    m = std::max(m, h[kRedBlocks + i]);
  }
  *mx = M;
  *mn = -m;
}

// ---------------------------------------------------------------------------
// NUFFT (exponential-of-semicircle kernel, upsampling 2)
// ---------------------------------------------------------------------------

constexpr int kW = 16;                  // kernel width (points)
constexpr double kBeta = 2.30 * kW;     // FINUFFT's beta for upsampling 2

__device__ __forceinline__ double es_phi(double z) {
  return fabs(z) <= 1.0 ? exp(kBeta * (sqrt(1.0 - z * z) - 1.0)) : 0.0;
}

// Gauss-Legendre nodes and weights on [-1, 1] (Newton on P_n)
static void gauss_legendre(int n, std::vector<double>& x,
                           std::vector<double>& w) {
  x.assign(n, 0.0);
  w.assign(n, 0.0);
  for (int i = 0; i < (n + 1) / 2; ++i) {
    double z = std::cos(M_PI * (i + 0.75) / (n + 0.5)), dp = 0.0;
    for (int it = 0; it < 100; ++it) {
      double p0 = 1.0, p1 = z;
      for (int k = 2; k <= n; ++k) {
        const double pk = ((2.0 * k - 1.0) * z * p1 - (k - 1.0) * p0) / k;
        p0 = p1;
        p1 = pk;
      }
      dp = n * (z * p1 - p0) / (z * z - 1.0);
      const double dz = p1 / dp;
      z -= dz;
      if (std::fabs(dz) < 1e-16) break;
    }
    x[i] = -z;
    x[n - 1 - i] = z;
    w[i] = w[n - 1 - i] = 2.0 / ((1.0 - z * z) * dp * dp);
  }
}

Nufft::Nufft(const double* h_angles, int P, int N, int nmodes)
    : P_(P), N_(N), nm_(nmodes) {
  TC_REQUIRE(P >= 1 && N >= 2 && nmodes >= 1, "FP64 NUFFT: bad geometry");
  nf_ = smooth_at_least(std::max(2 * nmodes, 2 * kW));
  if (nf_ % 2) nf_ = smooth_at_least(nf_ + 1);
  TC_REQUIRE(nf_ <= kMaxFFT,
             "FP64 NUFFT: fine grid of " + std::to_string(nf_) +
                 " points exceeds " + std::to_string(kMaxFFT) +
                 " (widths up to 2047 after padding)");
  std::vector<double2> cs(P);
  for (int p = 0; p < P; ++p)
    cs[p] = make_double2(std::cos(h_angles[p]), std::sin(h_angles[p]));
  // p(k) = h / psi_hat(k), psi_hat(k) = (w h / 2) int phi(z) cos(k z w h/2)
  const double h = 2.0 * M_PI / nf_;
  std::vector<double> zq, wq;
  gauss_legendre(200, zq, wq);
  std::vector<double> corr(nmodes);
  for (int i = 0; i < nmodes; ++i) {
    const int k = i - nmodes / 2;
    double integ = 0.0;
    for (size_t q = 0; q < zq.size(); ++q) {
      const double z = zq[q];
      const double ph = std::exp(kBeta * (std::sqrt(1.0 - z * z) - 1.0));
      integ += wq[q] * ph * std::cos(k * z * kW * h / 2.0);
    }
    corr[i] = h / ((kW * h / 2.0) * integ) * ((k & 1) ? -1.0 : 1.0);
  }
  std::vector<double> sx(P), sy(P);
  const double sc = (double)nf_ / (N - 1);
  for (int p = 0; p < P; ++p) {
    sx[p] = cs[p].x * sc;
    sy[p] = cs[p].y * sc;
  }
  ax_.alloc(sizeof(double) * P);
  ay_.alloc(sizeof(double) * P);
  TC_HIP(hipMemcpy(ax_.as<void>(), sx.data(), sizeof(double) * P,
                   hipMemcpyHostToDevice));
  TC_HIP(hipMemcpy(ay_.as<void>(), sy.data(), sizeof(double) * P,
                   hipMemcpyHostToDevice));
  cs_.alloc(sizeof(double2) * P);
  corr_.alloc(sizeof(double) * nmodes);
  TC_HIP(hipMemcpy(cs_.as<void>(), cs.data(), sizeof(double2) * P,
                   hipMemcpyHostToDevice));
  TC_HIP(hipMemcpy(corr_.as<void>(), corr.data(), sizeof(double) * nmodes,
                   hipMemcpyHostToDevice));
}

struct GridArgs {
  const double2* cs;
  int P, N, nf, S;
};

// fine-grid coordinate of point (p, j) along x (c.x) or y (c.y)
__device__ __forceinline__ void point_uv(const GridArgs& g, int p, int j,
                                         double* u, double* v) {
  const double2 c = g.cs[p];
  const double rr = (double)(j - g.N / 2) * ((double)g.nf / (g.N - 1));
  *u = rr * c.x + 0.5 * g.nf;
  *v = rr * c.y + 0.5 * g.nf;
}

// Type 1 on the FP64 matrix cores, with the FP32 kernel's scheme (spread_kernel
// in nufft.hip): a workgroup owns a tile and SB slices, a wave four regions of
// 4 x 16 cells, and v_mfma_f64_16x16x4 adds four points to a region and a slice
// pair.  Lane l holds row l / 16, column l % 16 and, in its four values, Re and
// Im of either slice (the FP64 product's rows are 4 v + l / 16 for value v).
// Every cell adds its points in list order: deterministic, where the atomic
// adds of the former kernel (512 an (slice, point)) were not.
// 2 x 200^2 at 150 angles: 1600 -> 54 us.
constexpr int kBatch = 128;
using f64x4 = __attribute__((__vector_size__(4 * sizeof(double)))) double;

struct SpreadArgs {
  TileGeom g;
  const double2* c;  // [S][P][N]
  double2* fine;     // [S][nf][nf]
  int S;
};

template <int SB>
__global__ void __launch_bounds__(64 * SP_WAVES)
spread_kernel(SpreadArgs a, const int4* __restrict__ work, double2* scratch) {
  constexpr int Q = SB / 2;
  constexpr int CS = 4 * Q + 1;
  // x weights at 1 .. 16, y weights at 18 .. 33, zeros at 0, 17 and 34: a cell
  // outside the footprint reads one of those
  __shared__ double pt_w[kBatch][35];
  __shared__ double pt_c[kBatch][CS];  // [Re, Im even slice, Re, Im odd][pair]
  __shared__ short2 pt_geo[kBatch];    // (index | l0x << 8, l0y)
  __shared__ int wlist[SP_WAVES][kBatch + 12];
  __shared__ int sg_off[kBatch + 1];
  __shared__ int2 sg[kBatch];
  __shared__ int sg_first;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lm = lane & 15, lk = lane >> 4;
  const int wi = xcd_remap(blockIdx.x, gridDim.x);
  const int4 item = work[2 * wi];
  const int4 segs = work[2 * wi + 1];  // the tile's segments [x, y)
  const int s0 = blockIdx.y * SB, ns = min(SB, a.S - s0);
  const TileWindow w = tile_window(a.g, item.x);
  const long sstride = (long)a.g.P * a.g.N;
  f64x4 acc[SP_REGIONS][Q];
#pragma unroll
  for (int g = 0; g < SP_REGIONS; ++g)
#pragma unroll
    for (int q = 0; q < Q; ++q) acc[g][q] = f64x4{0.0, 0.0, 0.0, 0.0};
  if (tid < kBatch) pt_w[tid][0] = pt_w[tid][17] = pt_w[tid][34] = 0.0;
  int seg = segs.x;
  if (item.y > 0) {
    // the segment that holds point f0 (offsets ascend from 0 at segs.x)
    for (int i = seg + tid; i < segs.y; i += 64 * SP_WAVES) {
      const int nxt = i + 1 < segs.y ? a.g.seg_off[i + 1] : 0x7fffffff;
      if (a.g.seg_off[i] <= item.y && item.y < nxt) sg_first = i;
    }
    __syncthreads();
    seg = sg_first;
  }
  const int pt = tid & (kBatch - 1);
  const int half = __builtin_amdgcn_readfirstlane(tid / kBatch);
  for (int fb0 = item.y; fb0 < item.z; fb0 += kBatch) {
    const int nb = min(kBatch, item.z - fb0);
    // the batch's segments: every segment has a point, so at most nb of them
    if (tid <= kBatch) {
      const int i = seg + tid;
      sg_off[tid] = i < segs.y ? a.g.seg_off[i] : 0x7fffffff;
      if (tid < kBatch) sg[tid] = i < segs.y ? a.g.seg[i] : make_int2(0, 0);
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
      const int lo = segment_of(f, kBatch);
      const int p = sg[lo].x, js = sg[lo].y;
      const int j = (js & 0xffff) + (f - sg_off[lo]);
      const double2* cp = a.c + (s0 + half) * sstride + (long)p * a.g.N + j;
      double2 cv[Q];
#pragma unroll
      for (int q = 0; q < Q; ++q)
        cv[q] = 2 * q + half < ns ? cp[2 * q * sstride] : make_double2(0., 0.);
      const double2 o = shift_origin(a.g, js >> 16);
      double frac;
      const int l0 = first_cell<kW>(half ? o.y : o.x, (double)(j - a.g.cidx),
                                    half ? a.g.ay[p] : a.g.ax[p], frac) -
                     (half ? w.Y0 : w.X0);  // -15 .. 31
      if (half)
        pt_geo[pt].y = (short)l0;
      else
        pt_geo[pt].x = (short)(pt | (l0 << 8));
      for (int m = 0; m < kW; ++m)
        pt_w[pt][17 * half + 1 + m] = es_phi((frac + m) * (2.0 / kW));
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        pt_c[pt][(2 * half) * Q + q] = cv[q].x;
        pt_c[pt][(2 * half + 1) * Q + q] = cv[q].y;
      }
      // the segment of the next batch's first point
      if (tid == nb - 1) sg_first = seg + segment_of(fb0 + nb, kBatch + 1);
    } else if (half == 0) {
      pt_geo[pt] = make_short2((short)(pt | (100 << 8)), 100);  // no region
    }
    __syncthreads();
    seg = sg_first;
#pragma unroll
    for (int g = 0; g < SP_REGIONS; ++g) {
      const int ry = region_y(wave, g), rx = region_x(wave, g);
      // points whose footprints meet the region, in point order: index and
      // footprint origin in the region, plus 16
      int cnt = 0;
#pragma unroll
      for (int c = 0; c < kBatch / 64; ++c) {
        const short2 e = pt_geo[c * 64 + lane];
        const int dx = (e.x >> 8) - rx, dy = e.y - ry;
        const bool hit = dx > -kW && dx < 16 && dy > -kW && dy < 4;
        const unsigned long long bal = __ballot(hit);
        const int pos =
            cnt + __builtin_amdgcn_mbcnt_hi((unsigned)(bal >> 32),
                                            __builtin_amdgcn_mbcnt_lo(
                                                (unsigned)bal, 0u));
        if (hit)
          wlist[wave][pos] = (e.x & 0xff) | (dx + 16) << 8 | (dy + 16) << 16;
        cnt += __popcll(bal);
      }
      if (cnt == 0) continue;
      // the last step and the look-ahead take a point of the batch with its
      // footprint out of reach
      if (lane < 12) wlist[wave][cnt + lane] = 0xffff00;
      __builtin_amdgcn_wave_barrier();
      for (int k0 = 0; k0 < cnt; k0 += 4) {
        const int e = wlist[wave][k0 + lk];
        const int i = e & 0xff;
        const int dx = min(max(lm + 16 - ((e >> 8) & 0xff), -1), kW);
        const int dy = min(max((lm & 3) + 16 - ((e >> 16) & 0xff), -1), kW);
        const double wx = pt_w[i][1 + dx], wy = pt_w[i][18 + dy];
#pragma unroll
        for (int q = 0; q < Q; ++q)
          acc[g][q] = __builtin_amdgcn_mfma_f64_16x16x4f64(
              wy * pt_c[i][(lm >> 2) * Q + q], wx, acc[g][q], 0, 0, 0);
      }
    }
    __syncthreads();  // the batch buffers are rewritten next
  }
  double2* dst = item.w < 0 ? nullptr
                            : scratch + ((long)item.w * gridDim.y +
                                         blockIdx.y) * (SB * SP_T * SP_T);
#pragma unroll
  for (int g = 0; g < SP_REGIONS; ++g) {
    const int ly = region_y(wave, g) + lk, lx = region_x(wave, g) + lm;
    const bool in = w.Y0 + ly < w.Y1 && w.X0 + lx < w.X1;
#pragma unroll
    for (int s = 0; s < SB; ++s) {
      const double2 val = make_double2(acc[g][s >> 1][2 * (s & 1)],
                                       acc[g][s >> 1][2 * (s & 1) + 1]);
      if (dst) {
        dst[(s * SP_T + ly) * SP_T + lx] = val;
      } else if (in && s < ns) {
        a.fine[((long)(s0 + s) * a.g.nf + w.Y0 + ly) * a.g.nf + w.X0 + lx] =
            val;
      }
    }
  }
}

// Adds the scratch slots of multi-chunk tiles into the fine grid, in slot
// order (deterministic): a quarter of a tile and a slice per workgroup, eight
// slots in flight.
__global__ void __launch_bounds__(256)
spread_fixup_kernel(SpreadArgs a, const int4* __restrict__ fix,
                    const double2* __restrict__ scratch, int sb) {
  const int4 f = fix[blockIdx.x];
  const int q = blockIdx.z >> 2, s = blockIdx.y * sb + q;
  if (s >= a.S) return;
  const TileWindow w = tile_window(a.g, f.x);
  const int cell = (blockIdx.z & 3) * 256 + threadIdx.x;
  const int ly = cell / SP_T, lx = cell - ly * SP_T;
  if (w.Y0 + ly >= w.Y1 || w.X0 + lx >= w.X1) return;
  const long slot_stride = (long)gridDim.y * sb * (SP_T * SP_T);
  const double2* base = scratch + (long)f.y * slot_stride +
                        ((long)blockIdx.y * sb + q) * (SP_T * SP_T) + cell;
  double2* o = a.fine + ((long)s * a.g.nf + w.Y0 + ly) * a.g.nf + w.X0 + lx;
  double2 sum = *o;
  constexpr int U = 8;
  for (int k = 0; k < f.z; k += U) {
    double2 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u)
      v[u] = k + u < f.z ? base[(long)(k + u) * slot_stride]
                         : make_double2(0.0, 0.0);
#pragma unroll
    for (int u = 0; u < U; ++u) sum = zadd(sum, v[u]);
  }
  *o = sum;
}

// type 2: sixteen lanes per (slice, point).  Lane b evaluates the weights of
// column and row b, gathers its column (a row's sixteen cells are contiguous)
// and the columns are summed over the lanes in a fixed order.  (One thread per
// point evaluated 32 exponentials and read single cells: 2 x 200^2 at 150 angles
// 65 -> 15 us.)
// The points are numbered from i0 on: a launch holds fewer than 2^32 threads
// (what is beyond is dropped without an error).
__global__ void __launch_bounds__(256)
interp_kernel(GridArgs g, const double2* __restrict__ fine, double2* c,
              long i0) {
  const long J = (long)g.P * g.N;
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long i = i0 + (t >> 4);
  const int b = (int)(t & 15);
  if (i >= J * g.S) return;  // all sixteen lanes of a point or none
  const int s = (int)(i / J);
  const long jj = i - (long)s * J;
  const int p = (int)(jj / g.N), j = (int)(jj - (long)p * g.N);
  double u, v;
  point_uv(g, p, j, &u, &v);
  const int lx = (int)ceil(u - 0.5 * kW), ly = (int)ceil(v - 0.5 * kW);
  const double wx = es_phi((lx + b - u) * (2.0 / kW));
  const double wy = es_phi((ly + b - v) * (2.0 / kW));
  int ix = (lx + b) % g.nf;
  if (ix < 0) ix += g.nf;
  const double2* f = fine + (long)s * g.nf * g.nf + ix;
  int iy = ly % g.nf;
  if (iy < 0) iy += g.nf;
  double2 q[kW];
#pragma unroll
  for (int a = 0; a < kW; ++a) {
    q[a] = f[(long)iy * g.nf];
    if (++iy == g.nf) iy = 0;
  }
  double2 acc = make_double2(0.0, 0.0);
#pragma unroll
  for (int a = 0; a < kW; ++a) {
    const double wa = __shfl(wy, a, 16);
    acc.x += wa * q[a].x;
    acc.y += wa * q[a].y;
  }
  acc.x *= wx;
  acc.y *= wx;
#pragma unroll
  for (int m = 8; m > 0; m >>= 1) {
    acc.x += __shfl_xor(acc.x, m, 16);
    acc.y += __shfl_xor(acc.y, m, 16);
  }
  if (b == 0) c[i] = acc;
}

// type 1 output: f[s][k2][k1] = corr(k1) corr(k2) fine[k2 mod nf][k1 mod nf]
__global__ void extract_kernel(const double2* __restrict__ fine,
                               const double* __restrict__ corr, int nm,
                               int nf, int S, double2* f, double* fr,
                               double rscale) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long per = (long)nm * nm;
  if (i >= per * S) return;
  const int s = (int)(i / per);
  const int rem = (int)(i - (long)s * per);
  const int i2 = rem / nm, i1 = rem - i2 * nm;
  int m1 = (i1 - nm / 2) % nf, m2 = (i2 - nm / 2) % nf;
  if (m1 < 0) m1 += nf;
  if (m2 < 0) m2 += nf;
  const double2 q = fine[((long)s * nf + m2) * nf + m1];
  const double w = corr[i1] * corr[i2];
  if (fr)
    fr[i] = q.x * w * rscale;
  else
    f[i] = make_double2(q.x * w, q.y * w);
}

// type 2 input: fine[k2 mod nf][k1 mod nf] = corr corr f (fine zeroed)
__global__ void place_kernel(const double* __restrict__ f,
                             const double* __restrict__ corr, int nm, int nf,
                             int S, double2* fine) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long per = (long)nm * nm;
  if (i >= per * S) return;
  const int s = (int)(i / per);
  const int rem = (int)(i - (long)s * per);
  const int i2 = rem / nm, i1 = rem - i2 * nm;
  int m1 = (i1 - nm / 2) % nf, m2 = (i2 - nm / 2) % nf;
  if (m1 < 0) m1 += nf;
  if (m2 < 0) m2 += nf;
  fine[((long)s * nf + m2) * nf + m1] =
      make_double2(f[i] * corr[i1] * corr[i2], 0.0);
}

void Nufft::type1(const double2* c, double2* f, double* fr, double rscale,
                  int S, hipStream_t s) {
  const long fplane = (long)nf_ * nf_;
  DevBuf grid(sizeof(double2) * (size_t)S * fplane);
  double2* fine = grid.as<double2>();
  SpreadArgs a{};
  a.g.ax = ax_.as<double>();
  a.g.ay = ay_.as<double>();
  a.g.P = P_;
  a.g.N = N_;
  a.g.cidx = N_ / 2;
  a.g.nf = a.g.ncols = nf_;
  a.g.ntx = (int)cdiv(nf_, SP_T);
  a.g.umax = (N_ / 2) * ((double)nf_ / (N_ - 1)) + 1.0;
  {
    // plans are shared by threads; the lists are built once, for good
    std::lock_guard<std::mutex> lk(mu_);
    if (!lists_ready_) {
      lists_.make_segments(a.g, kW, s);
      lists_.make_work(lists_.rule_chunk());
      TC_HIP(hipStreamSynchronize(s));  // other streams may read them next
      lists_ready_ = true;
    }
  }
  lists_.fill(a.g);
  // Groups of sb slices, as many to a launch as have their split tiles' scratch
  // slots in 1 GB, at most 65535.
  const int sb = S <= 2 ? 2 : 4;
  const size_t group_bytes = sizeof(double2) *
                             (size_t)std::max(lists_.nslots(), 1) * sb * SP_T *
                             SP_T;
  const int most = (int)std::max<size_t>(
      1, std::min<size_t>(65535, (size_t(1) << 30) / group_bytes));
  const int groups = std::min((int)cdiv(S, sb), most);
  DevBuf scratch(group_bytes * groups);
  auto k = sb == 2 ? spread_kernel<2> : spread_kernel<4>;
  for (int s0 = 0; s0 < S; s0 += groups * sb) {
    a.c = c + (long)s0 * P_ * N_;
    a.fine = fine + s0 * fplane;
    a.S = std::min(S - s0, groups * sb);
    const unsigned ng = cdiv(a.S, sb);
    hipLaunchKernelGGL(k, dim3((unsigned)lists_.nwork(), ng),
                       dim3(64 * SP_WAVES), 0, s, a, lists_.work(),
                       scratch.as<double2>());
    TC_HIP(hipGetLastError());
    if (lists_.nfix()) {
      hipLaunchKernelGGL(spread_fixup_kernel,
                         dim3((unsigned)lists_.nfix(), ng, 4 * sb), dim3(256),
                         0, s, a, lists_.fix(), scratch.as<double2>(), sb);
      TC_HIP(hipGetLastError());
    }
  }
  // only the columns of the modes are read back
  fft2(fine, S, nf_, nf_, +1, s, (nm_ + 1) / 2, nm_ / 2, false, true);
  const long nout = (long)S * nm_ * nm_;
  hipLaunchKernelGGL(extract_kernel, dim3(cdiv(nout, 256)), dim3(256), 0, s,
                     fine, corr_.as<double>(), nm_, nf_, S, f, fr, rscale);
  TC_HIP(hipGetLastError());
}

void Nufft::type2_real(const double* f, double2* c, int S, hipStream_t s) {
  const long fplane = (long)nf_ * nf_;
  DevBuf grid(sizeof(double2) * (size_t)S * fplane);
  double2* fine = grid.as<double2>();
  zero(fine, S * fplane, s);
  const long nin = (long)S * nm_ * nm_;
  hipLaunchKernelGGL(place_kernel, dim3(cdiv(nin, 256)), dim3(256), 0, s, f,
                     corr_.as<double>(), nm_, nf_, S, fine);
  TC_HIP(hipGetLastError());
  // rows without a mode are zero
  fft2(fine, S, nf_, nf_, -1, s, (nm_ + 1) / 2, nm_ / 2, true, false);
  GridArgs g{cs_.as<double2>(), P_, N_, nf_, S};
  const long npts = (long)S * P_ * N_, most = 1L << 27;
  for (long i0 = 0; i0 < npts; i0 += most) {
    hipLaunchKernelGGL(interp_kernel,
                       dim3(cdiv(16 * std::min(most, npts - i0), 256)),
                       dim3(256), 0, s, g, fine, c, i0);
    TC_HIP(hipGetLastError());
  }
}

// ---------------------------------------------------------------------------
// projectors: centred ray DFT fftshift(F(ifftshift v)) (src/gpu/fftshift.cu,
// src/fft.h) by direct summation: out[k] = sum_z v[z] w^(sign (z-c)(k-c)),
// c = N/2, w = exp(2 pi i / N)
// ---------------------------------------------------------------------------

template <bool IN_REAL, int SIGN, bool RAMP>
__global__ void ray_dft_kernel(const void* __restrict__ in, double2* out,
                               long nrays, int N,
                               const double2* __restrict__ tw) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nrays * N) return;
  const long ray = i / N;
  const int k = (int)(i - ray * N);
  const int c = N / 2;
  const long kk = k - c;
  double2 acc = make_double2(0.0, 0.0);
  for (int z = 0; z < N; ++z) {
    long m = ((long)(z - c) * kk) % N;
    if (m < 0) m += N;
    const double2 w = tw[m];  // exp(-2 pi i m / N)
    double2 x;
    if constexpr (IN_REAL)
      x = make_double2(reinterpret_cast<const double*>(in)[ray * N + z], 0.0);
    else
      x = reinterpret_cast<const double2*>(in)[ray * N + z];
    const double2 t = SIGN < 0 ? zmul(x, w) : zmulc(x, w);
    acc.x += t.x;
    acc.y += t.y;
  }
  if (RAMP) {
    const double r = fabs((double)(k - c)) / N;  // |k - N/2| / N (< 1)
    acc.x *= r;
    acc.y *= r;
  }
  out[i] = acc;
}

__global__ void real_part_kernel(const double2* __restrict__ in, double* out,
                                 long n, double scale) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = in[i].x * scale;
}

// Plans by geometry (device, sizes and the angles themselves): tables and
// lists only, no scratch, so threads and streams share them.  The 16 used last
// are kept; a caller's shared_ptr keeps a dropped one until it returns, and the
// release of its buffers (hipFree) waits for kernels that still read them.
static std::shared_ptr<Nufft> nufft_plan(const double* h_angles, int P, int N,
                                         int nmodes) {
  using Key = std::tuple<int, int, int, std::vector<double>>;
  static std::mutex mu;
  static std::list<std::pair<Key, std::shared_ptr<Nufft>>> plans;
  int dev = 0;
  TC_HIP(hipGetDevice(&dev));
  Key key(dev, N, nmodes, std::vector<double>(h_angles, h_angles + P));
  std::lock_guard<std::mutex> lk(mu);
  for (auto it = plans.begin(); it != plans.end(); ++it)
    if (it->first == key) {
      plans.splice(plans.begin(), plans, it);
      return plans.front().second;
    }
  ArenaPause no_arena;  // long-lived tables
  auto nu = std::make_shared<Nufft>(h_angles, P, N, nmodes);
  plans.emplace_front(std::move(key), nu);
  if (plans.size() > 16) plans.pop_back();
  return nu;
}

// Slices that the projectors take at once: their grids and samples within about
// 2 GB, in batches of one size.  The buffers are the calling thread's cached ones
// and stay after the call, so they must not grow with the stack.  (16 x 1400^2,
// 2.5 GB, gradient: 56.3 ms in two batches, 55.8 in one.)
static int slice_batch(int S, int P, int N, const Nufft& nu) {
  const double per = 16.0 * ((double)nu.nf() * nu.nf() + 2.0 * P * N);
  const int most = (int)std::max(1.0, std::min((double)S, 2.0e9 / per));
  const int n = (int)cdiv(S, most);
  return (int)cdiv(S, n);
}

void project(const double* img, double* sino, int S, int N,
             const double* h_angles, int P, hipStream_t s) {
  TC_REQUIRE(S >= 1 && N >= 2 && P >= 1, "FP64 project: bad shape");
  auto nu = nufft_plan(h_angles, P, N, N);
  const double2* tw = roots(N);
  const int B = slice_batch(S, P, N, *nu);
  const long rays = (long)P * N;  // samples of a slice
  DevBuf c(sizeof(double2) * B * rays), v(sizeof(double2) * B * rays);
  for (int s0 = 0; s0 < S; s0 += B) {
    const int nb = std::min(B, S - s0);
    const long ns = nb * rays;
    nu->type2_real(img + (long)s0 * N * N, c.as<double2>(), nb, s);
    hipLaunchKernelGGL((ray_dft_kernel<false, 1, false>), dim3(cdiv(ns, 256)),
                       dim3(256), 0, s, c.as<void>(), v.as<double2>(),
                       (long)nb * P, N, tw);
    TC_HIP(hipGetLastError());
    hipLaunchKernelGGL(real_part_kernel, dim3(cdiv(ns, 256)), dim3(256), 0, s,
                       v.as<double2>(), sino + s0 * rays, ns,
                       1.0 / ((double)N * N));
    TC_HIP(hipGetLastError());
  }
}

void backproject(const double* sino, double* img, int S, int P, int N,
                 const double* h_angles, bool fbp, hipStream_t s) {
  TC_REQUIRE(S >= 1 && N >= 2 && P >= 1, "FP64 backproject: bad shape");
  auto nu = nufft_plan(h_angles, P, N, N);
  const double2* tw = roots(N);
  const int B = slice_batch(S, P, N, *nu);
  const long rays = (long)P * N;
  DevBuf v(sizeof(double2) * B * rays);
  auto dft = fbp ? ray_dft_kernel<true, -1, true>
                 : ray_dft_kernel<true, -1, false>;
  for (int s0 = 0; s0 < S; s0 += B) {
    const int nb = std::min(B, S - s0);
    hipLaunchKernelGGL(dft, dim3(cdiv(nb * rays, 256)), dim3(256), 0, s,
                       (const void*)(sino + s0 * rays), v.as<double2>(),
                       (long)nb * P, N, tw);
    TC_HIP(hipGetLastError());
    nu->type1(v.as<double2>(), nullptr, img + (long)s0 * N * N,
              1.0 / ((double)N * N), nb, s);
  }
}

void gradient_nufft(const double* x, const double* b, double* g, int S, int N,
                    const double* h_angles, int P, hipStream_t s) {
  TC_REQUIRE(S >= 1 && N >= 2 && P >= 1, "FP64 gradient: bad shape");
  auto nu = nufft_plan(h_angles, P, N, N);
  const int B = slice_batch(S, P, N, *nu);
  const long img = (long)N * N;
  DevBuf c(sizeof(double2) * (size_t)B * P * N);
  for (int s0 = 0; s0 < S; s0 += B) {
    const int nb = std::min(B, S - s0);
    nu->type2_real(x + s0 * img, c.as<double2>(), nb, s);
    nu->type1(c.as<double2>(), nullptr, g + s0 * img,
              1.0 / ((double)N * N * N), nb, s);
  }
  if (b) axpby(g, b, g, S * img, 1.0, -1.0, s);
}

// ---------------------------------------------------------------------------
// Toeplitz operator
// ---------------------------------------------------------------------------

__global__ void psf_place_kernel(const double* __restrict__ psf, int n, int M,
                                 double2* circ) {
  const int n1 = 2 * n - 1;
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long)n1 * n1) return;
  const int a = (int)(i / n1), b = (int)(i - (long)a * n1);
  const int r = (a - (n - 1) + M) % M, c = (b - (n - 1) + M) % M;
  circ[(long)r * M + c] = make_double2(psf[i], 0.0);
}

Psf::Psf(const double* h_angles, int P, int n, hipStream_t s) : n_(n) {
  TC_REQUIRE(n >= 2 && P >= 1, "FP64 PSF: bad shape");
  M_ = smooth_at_least(2 * n - 1);
  TC_REQUIRE(M_ <= kMaxFFT, "FP64 PSF: width too large");
  const int n1 = 2 * n - 1;
  // PSF = Re(type 1 of ones) on (2n - 1)^2 modes (src/toeplitz.h:51-73)
  DevBuf ones(sizeof(double2) * (size_t)P * n), psf(sizeof(double) * n1 * n1);
  {
    std::vector<double2> h((size_t)P * n, make_double2(1.0, 0.0));
    TC_HIP(hipMemcpyAsync(ones.as<void>(), h.data(), sizeof(double2) * h.size(),
                          hipMemcpyHostToDevice, s));
    auto nu = nufft_plan(h_angles, P, n, n1);
    nu->type1(ones.as<double2>(), nullptr, psf.as<double>(), 1.0, 1, s);
    TC_HIP(hipStreamSynchronize(s));  // h leaves scope
  }
  spec_.alloc(sizeof(double2) * (size_t)M_ * M_);
  zero(spec_.as<double2>(), (long)M_ * M_, s);
  hipLaunchKernelGGL(psf_place_kernel, dim3(cdiv((long)n1 * n1, 256)),
                     dim3(256), 0, s, psf.as<double>(), n, M_,
                     spec_.as<double2>());
  TC_HIP(hipGetLastError());
  fft2(spec_.as<double2>(), 1, M_, M_, -1, s);
}

__global__ void pad_kernel(const double* __restrict__ x, int n, int M, int S,
                           double2* w) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long per = (long)M * M;
  if (i >= per * S) return;
  const int s = (int)(i / per);
  const int rem = (int)(i - (long)s * per);
  const int r = rem / M, c = rem - r * M;
  w[i] = make_double2(r < n && c < n ? x[((long)s * n + r) * n + c] : 0.0,
                      0.0);
}

__global__ void spec_mul_kernel(double2* w, const double2* __restrict__ h,
                                long per, int S) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= per * S) return;
  w[i] = zmul(w[i], h[i % per]);
}

// out = Re(w[0:n][0:n]) scale (- b)
__global__ void crop_kernel(const double2* __restrict__ w, int n, int M,
                            int S, double scale, const double* b,
                            double* out) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long per = (long)n * n;
  if (i >= per * S) return;
  const int s = (int)(i / per);
  const int rem = (int)(i - (long)s * per);
  const int r = rem / n, c = rem - r * n;
  const double v = w[((long)s * M + r) * M + c].x * scale;
  out[i] = b ? v - b[i] : v;
}

void Psf::apply(const double* x, const double* b, double* out, int S,
                hipStream_t s) {
  TC_REQUIRE(S >= 1, "FP64 Toeplitz: need at least one slice");
  const long per = (long)M_ * M_;
  // slices per group: about 1 GiB of complex workspace
  const int group = (int)std::max<long>(1, std::min<long>(S, (1L << 30) /
                                                                 (16 * per)));
  if ((size_t)group > work_slices_) {
    work_.alloc(sizeof(double2) * (size_t)group * per);
    work_slices_ = group;
  }
  double2* w = work_.as<double2>();
  const long img = (long)n_ * n_;
  const double scale = 1.0 / ((double)n_ * n_ * n_ * (double)M_ * M_);
  for (int s0 = 0; s0 < S; s0 += group) {
    const int ns = std::min(group, S - s0);
    hipLaunchKernelGGL(pad_kernel, dim3(cdiv(per * ns, 256)), dim3(256), 0, s,
                       x + s0 * img, n_, M_, ns, w);
    TC_HIP(hipGetLastError());
    fft2(w, ns, M_, M_, -1, s);
    hipLaunchKernelGGL(spec_mul_kernel, dim3(cdiv(per * ns, 256)), dim3(256),
                       0, s, w, spec_.as<double2>(), per, ns);
    TC_HIP(hipGetLastError());
    fft2(w, ns, M_, M_, +1, s);
    hipLaunchKernelGGL(crop_kernel, dim3(cdiv(img * ns, 256)), dim3(256), 0,
                       s, w, n_, M_, ns, scale, b ? b + s0 * img : nullptr,
                       out + s0 * img);
    TC_HIP(hipGetLastError());
  }
}

// ---------------------------------------------------------------------------
// qGGMRF (weights and rho' of src/gpu/potential_function.cuh:38-108)
// ---------------------------------------------------------------------------

constexpr double kMrfQ = 2.0, kMrfC = 0.001;

__device__ __forceinline__ double weight26(int dz, int dy, int dx) {
  const int k = (dz != 0) + (dy != 0) + (dx != 0);
  return k == 1 ? 0.0523 : (k == 2 ? 0.0370 : (k == 3 ? 0.0302 : 0.0));
}

// rho'(d) = sign(d) |d|^(q-1) / (sigma^q (c + t)) (q - (q - p) t / (c + t)),
// t = |d|^(q-p) / sigma^(q-p); rho'(0) = 0
__device__ __forceinline__ double d_rho(double d, double sigma, double p) {
  if (d == 0.0) return 0.0;
  const double ad = fabs(d);
  const double t1 = pow(ad, kMrfQ - p) / pow(sigma, kMrfQ - p);
  const double t2 = pow(ad, kMrfQ - 1.0);
  const double t3 = kMrfC + t1;
  const double mag = (t2 / (t3 * pow(sigma, kMrfQ))) *
                     (kMrfQ - ((kMrfQ - p) * t1) / t3);
  return d > 0.0 ? mag : -mag;
}

// rho(d) = |d/s|^q / (c + |d/s|^(q-p))
__device__ __forceinline__ double rho(double d, double sigma, double p) {
  const double u = fabs(d) / sigma;
  return pow(u, kMrfQ) / (kMrfC + pow(u, kMrfQ - p));
}

// FREE = false: neighbours clamped into the volume (the reference stencil);
// true: pairs leaving the volume are dropped
template <bool FREE>
__global__ void qggmrf_grad_kernel(const double* __restrict__ x, double* g,
                                   int S, int R, int C, double sigma,
                                   double p) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long per = (long)R * C;
  if (i >= per * S) return;
  const int s = (int)(i / per);
  const int rem = (int)(i - (long)s * per);
  const int r = rem / C, c = rem - r * C;
  const double v = x[i];
  double acc = 0.0;
  for (int dz = -1; dz <= 1; ++dz)
    for (int dy = -1; dy <= 1; ++dy)
      for (int dx = -1; dx <= 1; ++dx) {
        if (!dz && !dy && !dx) continue;
        int z = s + dz, y = r + dy, xx = c + dx;
        if (FREE) {
          if (z < 0 || z >= S || y < 0 || y >= R || xx < 0 || xx >= C)
            continue;
        } else {
          z = min(max(z, 0), S - 1);
          y = min(max(y, 0), R - 1);
          xx = min(max(xx, 0), C - 1);
        }
        acc += weight26(dz, dy, dx) *
               d_rho(v - x[((long)z * R + y) * C + xx], sigma, p);
      }
  g[i] += acc;
}

// 1/2 sum over in-bounds ordered pairs of w rho (free boundary), per block
__global__ void __launch_bounds__(256)
qggmrf_value_kernel(const double* __restrict__ x, int S, int R, int C,
                    double sigma, double p, double* part) {
  __shared__ double red[256];
  const long per = (long)R * C;
  double acc = 0.0;
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < per * S;
       i += (long)gridDim.x * 256) {
    const int s = (int)(i / per);
    const int rem = (int)(i - (long)s * per);
    const int r = rem / C, c = rem - r * C;
    const double v = x[i];
    for (int dz = -1; dz <= 1; ++dz)
      for (int dy = -1; dy <= 1; ++dy)
        for (int dx = -1; dx <= 1; ++dx) {
          if (!dz && !dy && !dx) continue;
          const int z = s + dz, y = r + dy, xx = c + dx;
          if (z < 0 || z >= S || y < 0 || y >= R || xx < 0 || xx >= C)
            continue;
          acc += weight26(dz, dy, dx) *
                 rho(v - x[((long)z * R + y) * C + xx], sigma, p);
        }
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = 0.5 * red[0];
}

void add_total_var(const double* x, double* g, int S, int R, int C,
                   double sigma, double p, hipStream_t s) {
  TC_REQUIRE(S >= 1 && R >= 1 && C >= 1 && sigma > 0.0, "FP64 qGGMRF: bad "
                                                        "arguments");
  const long n = (long)S * R * C;
  hipLaunchKernelGGL(qggmrf_grad_kernel<false>, dim3(cdiv(n, 256)), dim3(256),
                     0, s, x, g, S, R, C, sigma, p);
  TC_HIP(hipGetLastError());
}

void add_qggmrf_grad_free(const double* x, double* g, int S, int R, int C,
                          double sigma, double p, hipStream_t s) {
  TC_REQUIRE(S >= 1 && R >= 1 && C >= 1 && sigma > 0.0, "FP64 qGGMRF: bad "
                                                        "arguments");
  const long n = (long)S * R * C;
  hipLaunchKernelGGL(qggmrf_grad_kernel<true>, dim3(cdiv(n, 256)), dim3(256),
                     0, s, x, g, S, R, C, sigma, p);
  TC_HIP(hipGetLastError());
}

double qggmrf_value_free(const double* x, int S, int R, int C, double sigma,
                         double p, hipStream_t s) {
  TC_REQUIRE(S >= 1 && R >= 1 && C >= 1 && sigma > 0.0, "FP64 qGGMRF: bad "
                                                        "arguments");
  DevBuf part(sizeof(double) * (kRedBlocks + 1));
  hipLaunchKernelGGL(qggmrf_value_kernel, dim3(kRedBlocks), dim3(256), 0, s,
                     x, S, R, C, sigma, p, part.as<double>());
  TC_HIP(hipGetLastError());
  return reduce_host(part.as<double>(), kRedBlocks, s);
}

// ---------------------------------------------------------------------------
// pre/post-processing (src/preproc.cpp:62-108, src/postproc.cpp:69-102,
// src/gpu/padding.cu:119-150)
// ---------------------------------------------------------------------------

__global__ void preproc_kernel(const double* __restrict__ in, double* out,
                               long rows, int N, int N2, int npad, int off,
                               double scale, double shift) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= rows * N2) return;
  const long r = idx / N2;
  const int z = (int)(idx - r * N2);
  int zs = (z + off) % N2;
  if (zs < 0) zs += N2;
  const int zi = zs - npad;
  out[idx] = (zi >= 0 && zi < N) ? (in[r * N + zi] - shift) * scale : 0.0;
}

__global__ void pad2d_kernel(const double* __restrict__ in, double* out,
                             int S, int nin, int nout, int shift) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long per = (long)nout * nout;
  if (idx >= per * S) return;
  const long s = idx / per;
  const int rem = (int)(idx - s * per);
  const int r = rem / nout - shift, c = rem - (rem / nout) * nout - shift;
  out[idx] = (r >= 0 && r < nin && c >= 0 && c < nin)
                 ? in[(s * nin + r) * nin + c]
                 : 0.0;
}

__global__ void crop2d_kernel(const double* __restrict__ in, double* out,
                              int S, int nin, int nout, int shift) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long per = (long)nout * nout;
  if (idx >= per * S) return;
  const long s = idx / per;
  const int rem = (int)(idx - s * per);
  const int r = rem / nout, c = rem - r * nout;
  out[idx] = in[(s * nin + r + shift) * nin + c + shift];
}

static void pad_to(const double* in, double* out, int S, int nin, int nout,
                   hipStream_t s) {
  const long n = (long)S * nout * nout;
  hipLaunchKernelGGL(pad2d_kernel, dim3(cdiv(n, 256)), dim3(256), 0, s, in,
                     out, S, nin, nout, (nout - nin) / 2);
  TC_HIP(hipGetLastError());
}

static void crop2d(const double* in, double* out, int S, int nin, int nout,
                   hipStream_t s) {
  const long n = (long)S * nout * nout;
  hipLaunchKernelGGL(crop2d_kernel, dim3(cdiv(n, 256)), dim3(256), 0, s, in,
                     out, S, nin, nout, (nin - nout) / 2);
  TC_HIP(hipGetLastError());
}

// src/preproc.cpp:75-86 with the centre in FP64
static void pad_amount64(int nrays, double center, int* npad, int* offset) {
  const int cen = (int)std::round(center);  // halves away from zero
  const int off = (nrays + 1) / 2 - cen;
  int np = static_cast<int>(0.42 * nrays) / 2;
  if (std::abs(off) > np) np = std::abs(off);
  *npad = np;
  *offset = off;
}

int preproc(const double* in, double* out, int S, int P, int N, double center,
            hipStream_t s) {
  int npad = 0, off = 0;
  pad_amount64(N, center, &npad, &off);
  if (!out) return npad;
  TC_REQUIRE(in != nullptr, "null argument");
  const int n2 = N + 2 * npad;
  const long n = (long)S * P * n2;
  hipLaunchKernelGGL(preproc_kernel, dim3(cdiv(n, 256)), dim3(256), 0, s, in,
                     out, (long)S * P, N, n2, npad, off, 1.0, 0.0);
  TC_HIP(hipGetLastError());
  return npad;
}

void postproc(const double* in, double* out, int S, int nin, int nout,
              hipStream_t s) {
  TC_REQUIRE(nout >= 1 && nout <= nin, "postproc: bad shape");
  crop2d(in, out, S, nin, nout, s);
}

void pad2d(const double* in, double* out, int S, int nin, int padding,
           hipStream_t s) {
  TC_REQUIRE(S >= 1 && nin >= 1, "pad2d: bad shape");
  pad_to(in, out, S, nin, nin + std::abs(padding), s);
}

__global__ void __launch_bounds__(256)
diff2_kernel(const double* a, const double* b, long n, double* part) {
  __shared__ double red[256];
  double acc = 0.0;
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n;
       i += (long)gridDim.x * 256) {
    const double d = a[i] - b[i];
    acc += d * d;
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

double diff_norm2(const double* a, const double* b, long n, hipStream_t s) {
  DevBuf part(sizeof(double) * (kRedBlocks + 1));
  hipLaunchKernelGGL(diff2_kernel, dim3(kRedBlocks), dim3(256), 0, s, a, b, n,
                     part.as<double>());
  TC_HIP(hipGetLastError());
  return reduce_host(part.as<double>(), kRedBlocks, s);
}

// ---------------------------------------------------------------------------
// Optimizer::run2 (src/optimize.h:96-154) on device-resident FP64 state, with
// one operator application per attempt: gradient(y) = Ay - b + R'(y) for a
// linear A, and err(v) from a quadratic form (Toeplitz: ||y||^2 + v.Av -
// 2 v.b) or the projector (||Pv - y||)
// ---------------------------------------------------------------------------

struct Run2Ops {
  std::function<void(const double*, double*)> A;  // out = A v
  // err(v) given v and A v; for the projector form A v is unused
  std::function<double(const double*, const double*)> err;
};

static int run2(const Run2Ops& ops, const double* x0, const double* b,
                double* out, long N, int S, int R, int C, int num_iters,
                double step0, double sigma, double p, double* last_err,
                int* attempts, hipStream_t s) {
  DevBuf bs(sizeof(double) * N), bx(sizeof(double) * N),
      bTs(sizeof(double) * N), bTx(sizeof(double) * N),
      by(sizeof(double) * N), bTy(sizeof(double) * N), bg(sizeof(double) * N),
      bTg(sizeof(double) * N);
  double *sol = bs.as<double>(), *x = bx.as<double>(), *Ts = bTs.as<double>(),
         *Tx = bTx.as<double>(), *y = by.as<double>(), *Ty = bTy.as<double>(),
         *g = bg.as<double>(), *Tg = bTg.as<double>();
  TC_HIP(hipMemcpyAsync(sol, x0, sizeof(double) * N, hipMemcpyDeviceToDevice,
                        s));
  TC_HIP(hipMemcpyAsync(x, x0, sizeof(double) * N, hipMemcpyDeviceToDevice,
                        s));
  ops.A(sol, Ts);
  TC_HIP(hipMemcpyAsync(Tx, Ts, sizeof(double) * N, hipMemcpyDeviceToDevice,
                        s));
  double t = 1.0, tnew = 1.0, step = step0, fx = 0.0;
  int it = 0, att = 0;
  for (; it < num_iters; ++it) {
    for (;;) {
      const double beta = tnew * (1.0 / t - 1.0);
      tnew = 0.5 * (std::sqrt(t * t * t * t + 4.0 * t * t) - t * t);
      // y = sol + beta (sol - x), T y likewise (linearity)
      axpby(sol, x, y, N, 1.0 + beta, -beta, s);
      axpby(Ts, Tx, Ty, N, 1.0 + beta, -beta, s);
      // g = T y - b + R'(y)
      axpby(Ty, b, g, N, 1.0, -1.0, s);
      add_total_var(y, g, S, R, C, sigma, p, s);
      ops.A(g, Tg);
      // candidate and its image under A
      axpby(y, g, sol, N, 1.0, -step, s);
      axpby(Ty, Tg, Ts, N, 1.0, -step, s);
      ++att;
      fx = ops.err(sol, Ts);
      const double fy = ops.err(y, Ty);
      const double gy = 0.5 * step * dot(g, g, N, s);
      if (fx > fy + gy) {
        step *= 0.9;
        continue;
      }
      TC_HIP(hipMemcpyAsync(x, sol, sizeof(double) * N,
                            hipMemcpyDeviceToDevice, s));
      TC_HIP(hipMemcpyAsync(Tx, Ts, sizeof(double) * N,
                            hipMemcpyDeviceToDevice, s));
      step = step0;
      t = tnew;
      break;
    }
  }
  TC_HIP(hipMemcpyAsync(out, sol, sizeof(double) * N, hipMemcpyDeviceToDevice,
                        s));
  TC_HIP(hipStreamSynchronize(s));
  if (last_err) *last_err = fx;
  if (attempts) *attempts = att;
  return it;
}

Result mbir2(const double* sino, const double* x0, double* recon, int S,
             int P, int N, const double* h_angles, double center,
             int num_iters, double sigma, double p, hipStream_t s) {
  TC_REQUIRE(S >= 1 && P >= 1 && N >= 2, "FP64 mbir2: bad sinogram shape");
  TC_REQUIRE(h_angles != nullptr, "FP64 mbir2: null angles");
  TC_REQUIRE(num_iters >= 0, "FP64 mbir2: num_iters must be >= 0");
  ArenaScope arena;
  Result res;
  const long nsino = (long)S * P * N;
  const size_t img_b = sizeof(double) * (size_t)S * N * N;
  double mx = 0.0, mn = 0.0;
  minmax(sino, nsino, &mx, &mn, s);
  res.max_sino = mx;
  if (mx == 0.0) {
    if (!x0) throw Error(TC_ERR_VALUE, "mbir2: sinogram has ZERO max value");
    TC_HIP(hipMemcpyAsync(recon, x0, img_b, hipMemcpyDeviceToDevice, s));
    TC_HIP(hipStreamSynchronize(s));
    return res;
  }
  // normalise (src/mbir2.cpp:46-54) and the FBP guess (:56-60)
  DevBuf bs2(sizeof(double) * nsino);
  axpby(sino, nullptr, bs2.as<double>(), nsino, 1.0 / mx, 0.0, s);
  DevBuf bx0(img_b);
  if (x0)
    TC_HIP(hipMemcpyAsync(bx0.as<void>(), x0, img_b, hipMemcpyDeviceToDevice,
                          s));
  else
    backproject(bs2.as<double>(), bx0.as<double>(), S, P, N, h_angles, true,
                s);
  // pad and centre (:63-66)
  int npad = 0, off = 0;
  pad_amount64(N, center, &npad, &off);
  const int n2 = N + 2 * npad;
  res.padded = n2;
  const long ns2 = (long)S * P * n2;
  DevBuf bsp(sizeof(double) * ns2);
  hipLaunchKernelGGL(preproc_kernel, dim3(cdiv(ns2, 256)), dim3(256), 0, s,
                     bs2.as<double>(), bsp.as<double>(), (long)S * P, N, n2,
                     npad, off, 1.0, 0.0);
  TC_HIP(hipGetLastError());
  const long nimg = (long)S * n2 * n2;
  DevBuf bx0p(sizeof(double) * nimg), bb(sizeof(double) * nimg);
  pad_to(bx0.as<double>(), bx0p.as<double>(), S, N, n2, s);
  // b = P^T y, ||y||^2 (:74-77)
  backproject(bsp.as<double>(), bb.as<double>(), S, P, n2, h_angles, false,
              s);
  res.sino_norm = dot(bsp.as<double>(), bsp.as<double>(), ns2, s);
  // PSF (:86-97) and L = max(T 1) (:101-112)
  Psf psf(h_angles, P, n2, s);
  {
    const long nn = (long)n2 * n2;
    DevBuf ones(sizeof(double) * nn), t1(sizeof(double) * nn);
    hipLaunchKernelGGL(fill_kernel, dim3(cdiv(nn, 256)), dim3(256), 0, s,
                       ones.as<double>(), nn, 1.0);
    TC_HIP(hipGetLastError());
    psf.apply(ones.as<double>(), nullptr, t1.as<double>(), 1, s);
    double lmin = 0.0;
    minmax(t1.as<double>(), nn, &res.lipschitz, &lmin, s);
  }
  res.step = std::min(1.0, 1.0 / res.lipschitz);
  const double yd2 = res.sino_norm;
  const double* b = bb.as<double>();
  Run2Ops ops;
  ops.A = [&](const double* v, double* out) {
    psf.apply(v, nullptr, out, S, s);
  };
  // err(v) = sqrt(||y||^2 + v.Tv - 2 v.b) (src/error2.cpp:60-63,91)
  ops.err = [&](const double* v, const double* Tv) {
    return std::sqrt(yd2 + dot(v, Tv, nimg, s) - 2.0 * dot(v, b, nimg, s));
  };
  DevBuf bsol(sizeof(double) * nimg);
  res.iterations = run2(ops, bx0p.as<double>(), b, bsol.as<double>(), nimg, S,
                        n2, n2, num_iters, res.step, sigma, p,
                        &res.last_error, &res.attempts, s);
  crop2d(bsol.as<double>(), recon, S, n2, N, s);
  TC_HIP(hipStreamSynchronize(s));
  return res;
}

Result mbir_nufft(const double* sino, const double* x0, double* recon, int S,
                  int P, int N, const double* h_angles, double center,
                  int num_iters, double sigma, double p, hipStream_t s) {
  TC_REQUIRE(S >= 1 && P >= 1 && N >= 2, "FP64 mbir: bad sinogram shape");
  TC_REQUIRE(h_angles != nullptr && x0 != nullptr,
             "FP64 mbir: angles and an initial guess are required");
  TC_REQUIRE(num_iters >= 0, "FP64 mbir: num_iters must be >= 0");
  ArenaScope arena;
  Result res;
  const long nsino = (long)S * P * N;
  const size_t img_b = sizeof(double) * (size_t)S * N * N;
  double mx = 0.0, mn = 0.0;
  minmax(sino, nsino, &mx, &mn, s);
  res.max_sino = mx;
  if (mx == mn) {
    TC_HIP(hipMemcpyAsync(recon, x0, img_b, hipMemcpyDeviceToDevice, s));
    TC_HIP(hipStreamSynchronize(s));
    return res;
  }
  // normalise to [0, 1] and pad (src/mbir.cpp:43-60)
  int npad = 0, off = 0;
  pad_amount64(N, center, &npad, &off);
  const int n2 = N + 2 * npad;
  res.padded = n2;
  const long ns2 = (long)S * P * n2;
  DevBuf bsp(sizeof(double) * ns2);
  hipLaunchKernelGGL(preproc_kernel, dim3(cdiv(ns2, 256)), dim3(256), 0, s,
                     sino, bsp.as<double>(), (long)S * P, N, n2, npad, off,
                     1.0 / (mx - mn), mn);
  TC_HIP(hipGetLastError());
  const long nimg = (long)S * n2 * n2;
  DevBuf bx0p(sizeof(double) * nimg), bb(sizeof(double) * nimg);
  pad_to(x0, bx0p.as<double>(), S, N, n2, s);
  backproject(bsp.as<double>(), bb.as<double>(), S, P, n2, h_angles, false,
              s);
  res.sino_norm = dot(bsp.as<double>(), bsp.as<double>(), ns2, s);
  {
    const long nn = (long)n2 * n2;
    DevBuf ones(sizeof(double) * nn), t1(sizeof(double) * nn);
    hipLaunchKernelGGL(fill_kernel, dim3(cdiv(nn, 256)), dim3(256), 0, s,
                       ones.as<double>(), nn, 1.0);
    TC_HIP(hipGetLastError());
    gradient_nufft(ones.as<double>(), nullptr, t1.as<double>(), 1, n2,
                   h_angles, P, s);
    double lmin = 0.0;
    minmax(t1.as<double>(), nn, &res.lipschitz, &lmin, s);
  }
  res.step = std::min(1.0, 1.0 / res.lipschitz);
  DevBuf bproj(sizeof(double) * ns2);
  Run2Ops ops;
  ops.A = [&](const double* v, double* out) {
    gradient_nufft(v, nullptr, out, S, n2, h_angles, P, s);
  };
  // err(v) = ||P v - y|| (src/error.cpp:57-59)
  ops.err = [&](const double* v, const double*) {
    project(v, bproj.as<double>(), S, n2, h_angles, P, s);
    axpby(bproj.as<double>(), bsp.as<double>(), bproj.as<double>(), ns2, 1.0,
          -1.0, s);
    return std::sqrt(dot(bproj.as<double>(), bproj.as<double>(), ns2, s));
  };
  DevBuf bsol(sizeof(double) * nimg);
  res.iterations = run2(ops, bx0p.as<double>(), bb.as<double>(),
                        bsol.as<double>(), nimg, S, n2, n2, num_iters,
                        res.step, sigma, p, &res.last_error, &res.attempts, s);
  crop2d(bsol.as<double>(), recon, S, n2, N, s);
  TC_HIP(hipStreamSynchronize(s));
  return res;
}

}  // namespace f64
}  // namespace tc
