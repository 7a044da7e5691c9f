// Host plans and the generic batched line FFT kernel.
#include <cmath>
#include <cstdlib>
#include <functional>
#include <map>
#include <memory>
#include <mutex>
#include <tuple>

#include "fft_ops.h"
#include "fft_rt.h"
#include "lds_launch.h"

namespace tc {

std::vector<int> fft_factor(int L) {
  TC_REQUIRE(L >= 1, "FFT length must be positive");
  std::vector<int> r;
  int m = L;
  int p2 = 0;
  while (m % 2 == 0) {
    m /= 2;
    ++p2;
  }
  while (p2 >= 3) {
    r.push_back(8);
    p2 -= 3;
  }
  if (p2 == 2) r.push_back(4);
  if (p2 == 1) r.push_back(2);
  for (int p : {3, 5, 7}) {
    while (m % p == 0) {
      r.push_back(p);
      m /= p;
    }
  }
  TC_REQUIRE(m == 1, "FFT length " + std::to_string(L) +
                         " is not a product of 2, 3, 5, 7");
  TC_REQUIRE((int)r.size() <= FFT_MAX_STAGES, "FFT length too large");
  return r;
}

bool fft_smooth(int L) {
  if (L < 1) return false;
  for (int p : {2, 3, 5, 7})
    while (L % p == 0) L /= p;
  return L == 1;
}

int fft_next_smooth(int n, bool even) {
  int m = n < 1 ? 1 : n;
  for (;; ++m) {
    if (even && (m % 2)) continue;
    if (fft_smooth(m)) return m;
  }
}

// The radices of L: as few stages as possible, and of those the largest
// smallest radix (so that the stages have alike numbers of butterflies).
static std::vector<int> rt_factor(int L) {
  static const int kRadices[] = {16, 15, 14, 12, 10, 9, 8, 7, 6, 5, 4, 3, 2};
  std::vector<int> best, cur;
  std::function<void(int, int)> go = [&](int m, int from) {
    if (!best.empty() && cur.size() >= best.size() && m > 1) return;
    if (m == 1) {
      if (best.empty() || cur.size() < best.size() ||
          (cur.size() == best.size() && cur.back() > best.back()))
        best = cur;
      return;
    }
    for (int i = from; i < 13; ++i)
      if (m % kRadices[i] == 0) {
        cur.push_back(kRadices[i]);
        go(m / kRadices[i], i);
        cur.pop_back();
      }
  };
  go(L, 0);
  TC_REQUIRE(L == 1 || !best.empty(), "FFT length " + std::to_string(L) +
                                          " is not a product of 2, 3, 5, 7");
  TC_REQUIRE((int)best.size() <= RT_MAX_STAGES, "FFT length too large");
  return best;
}

FFTLength::FFTLength(int L) {
  ArenaPause no_arena;  // process-lifetime table, filled synchronously
  std::vector<int> r = fft_factor(L);
  radices_ = rt_factor(L);
  plan_.L = L;
  plan_.nst = (int)r.size();
  for (int i = 0; i < plan_.nst; ++i) plan_.radix[i] = r[i];
  std::vector<float2> h(L);
  for (int m = 0; m < L; ++m) {
    double a = -2.0 * M_PI * (double)m / (double)L;
    h[m] = make_float2((float)std::cos(a), (float)std::sin(a));
  }
  tw_.alloc(sizeof(float2) * L);
  TC_HIP(hipMemcpy(tw_.as<void>(), h.data(), sizeof(float2) * L,
                   hipMemcpyHostToDevice));
  plan_.tw = tw_.as<float2>();
}

int FFTLength::min_radix() const {
  int m = 8;
  for (int i = 0; i < plan_.nst; ++i) m = std::min(m, plan_.radix[i]);
  return plan_.nst ? m : 1;
}

int FFTLength::nb_for(int nlines, int nthr) const {
  long need = (long)nlines * (plan_.L / min_radix());
  long nb = (need + nthr - 1) / nthr;
  if (nb <= 1) return 1;
  if (nb <= 2) return 2;
  if (nb <= 4) return 4;
  if (nb <= 8) return 8;
  return 0;  // not supported
}

const FFTLength& fft_length(int L) {
  static std::mutex mu;
  static std::map<std::pair<int, int>, std::unique_ptr<FFTLength>> cache;
  int dev = 0;
  TC_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lk(mu);
  auto key = std::make_pair(dev, L);
  auto it = cache.find(key);
  if (it == cache.end())
    it = cache.emplace(key, std::make_unique<FFTLength>(L)).first;
  return *it->second;
}

const float2* fft_stage_twiddles(const std::vector<int>& a,
                                 const std::vector<int>& b) {
  using Key = std::tuple<int, std::vector<int>, std::vector<int>>;
  static std::mutex mu;
  static std::map<Key, std::unique_ptr<DevBuf>> cache;
  int dev = 0;
  TC_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lk(mu);
  Key key(dev, a, b);
  auto it = cache.find(key);
  if (it == cache.end()) {
    ArenaPause no_arena;  // process-lifetime table, filled synchronously
    std::vector<float2> h;
    for (const std::vector<int>* rs : {&a, &b}) {
      long L = 1, Ns = 1;
      for (int r : *rs) L *= r;
      for (size_t s = 0; s < rs->size(); ++s) {
        const int R = (*rs)[s];
        const long step = L / (Ns * R);
        if (s > 0)
          for (int r = 1; r < R; ++r)
            for (long k = 0; k < Ns; ++k) {
              const double x = -2.0 * M_PI * (double)(k * r * step) / (double)L;
              h.push_back(make_float2((float)std::cos(x), (float)std::sin(x)));
            }
        Ns *= R;
      }
    }
    if (h.empty()) h.push_back(make_float2(1.f, 0.f));
    auto buf = std::make_unique<DevBuf>(sizeof(float2) * h.size());
    TC_HIP(hipMemcpy(buf->as<void>(), h.data(), sizeof(float2) * h.size(),
                     hipMemcpyHostToDevice));
    it = cache.emplace(std::move(key), std::move(buf)).first;
  }
  return it->second->as<float2>();
}

// bytes of LDS of lpw lines in two buffers
static size_t rt_bytes(int L, int lpw) {
  return 2 * sizeof(float2) * (size_t)lpw * (rt_pad(L) + 1);
}
bool rt_fits(int L) { return rt_bytes(L, 1) <= 160 * 1024; }

RtLaunch rt_launch(int L, long nlines, int want) {
  TC_REQUIRE(rt_fits(L), "FFT line does not fit in LDS");
  const FFTLength& F = fft_length(L);
  RtLaunch l;
  l.plan.L = L;
  l.plan.tw = F.plan().tw;
  l.plan.nst = (int)F.radices().size();
  for (int i = 0; i < l.plan.nst; ++i) l.plan.radix[i] = F.radices()[i];
  l.plan.ldl = rt_pad(L) + 1;
  l.lpw = 1;
  while (2 * l.lpw <= want && rt_bytes(L, 2 * l.lpw) <= 64 * 1024 &&
         nlines > l.lpw)
    l.lpw *= 2;
  l.plan.lines_off = l.lpw * l.plan.ldl;
  const int rmin = l.plan.nst ? F.radices().back() : 1;
  const long nb = (long)l.lpw * L / rmin;
  l.nthr = (int)std::min<long>(RT_MAX_THREADS, (nb + 63) / 64 * 64);
  l.smem = rt_bytes(L, l.lpw);
  return l;
}

// Line l of batch b starts at b*bstride + (l/lgroup)*lstride + l%lgroup,
// element i at + i*estride
// (complex elements).  Of a line, the elements [0, nin) and [L - nin_hi, L)
// are read (the others are zero) and [0, nout) and [L - nout_hi, L) written.
struct LinesMap {
  int lines_per_batch, nin, nin_hi, nout, nout_hi, colmajor, lgroup;
  long total, bstride, lstride, estride;
  float scale;
};

__device__ __forceinline__ long line_base(const LinesMap& m, long gl) {
  const long b = gl / m.lines_per_batch;
  const int l = (int)(gl - b * m.lines_per_batch);
  return b * m.bstride + (l / m.lgroup) * m.lstride + l % m.lgroup;
}

template <int DIR>
__global__ void __launch_bounds__(RT_MAX_THREADS)
rt_lines_kernel(const float2* __restrict__ in, float2* __restrict__ out,
                RtPlan P, LinesMap m, int lpw) {
  extern __shared__ float2 sm[];
  const int tid = threadIdx.x, nthr = blockDim.x, L = P.L;
  const long l0 = (long)blockIdx.x * lpw;
  const int nl = (int)min((long)lpw, m.total - l0);
  for (int t = tid; t < lpw * L; t += nthr) {
    const int l = m.colmajor ? t % lpw : t / L;
    const int i = m.colmajor ? t / lpw : t - l * L;
    float2 v = make_float2(0.f, 0.f);
    if (l < nl && (i < m.nin || i >= L - m.nin_hi))
      v = in[line_base(m, l0 + l) + (long)i * m.estride];
    sm[l * P.ldl + rt_pad(i)] = v;
  }
  __syncthreads();
  const float2* z = rt_fft<DIR>(sm, lpw, P, tid, nthr);
  const int nw = m.nout + m.nout_hi;  // elements written per line
  for (int t = tid; t < lpw * nw; t += nthr) {
    const int l = m.colmajor ? t % lpw : t / nw;
    int i = m.colmajor ? t / lpw : t - l * nw;
    if (i >= m.nout) i += L - nw;
    if (l < nl)
      out[line_base(m, l0 + l) + (long)i * m.estride] =
          cscale(z[l * P.ldl + rt_pad(i)], m.scale);
  }
}

// lines of more than rt_fits() points: one line per workgroup, in place
template <int DIR, int NB>
__global__ void __launch_bounds__(1024)
fft_lines_kernel(const float2* __restrict__ in, float2* __restrict__ out,
                 FFTPlan P, LinesMap m) {
  extern __shared__ float2 sm[];
  const int tid = threadIdx.x, nthr = blockDim.x, L = P.L;
  const long base = line_base(m, blockIdx.x);
  for (int i = tid; i < L; i += nthr)
    sm[i] = (i < m.nin || i >= L - m.nin_hi) ? in[base + (long)i * m.estride]
                                             : make_float2(0.f, 0.f);
  __syncthreads();
  fft_lds<DIR, NB>(sm, 1, L, P, tid, nthr);
  const int nw = m.nout + m.nout_hi;
  for (int t = tid; t < nw; t += nthr) {
    const int i = t < m.nout ? t : t + L - nw;
    out[base + (long)i * m.estride] = cscale(sm[i], m.scale);
  }
}

template <int DIR>
static void launch_lines(const LineFFTArgs& a, hipStream_t stream) {
  LinesMap m{a.lines_per_batch, a.nin,     a.nin_hi,  a.nout,
             a.nout_hi,         a.colmajor, a.lgroup,
             (long)a.lines_per_batch * a.nbatch,
             a.bstride,         a.lstride, a.estride, a.scale};
  if (m.total == 0) return;
  if (rt_fits(a.L)) {
    const RtLaunch l = rt_launch(a.L, m.total, a.colmajor ? 16 : 4);
    auto k = rt_lines_kernel<DIR>;
    allow_lds((const void*)k, l.smem);
    hipLaunchKernelGGL(k, dim3(cdiv(m.total, l.lpw)), dim3(l.nthr), l.smem,
                       stream, a.in, a.out, l.plan, m, l.lpw);
    TC_HIP(hipGetLastError());
    return;
  }
  const FFTLength& F = fft_length(a.L);
  const size_t smem = sizeof(float2) * (size_t)a.L;
  const int nb = F.nb_for(1, 1024);
  TC_REQUIRE(smem <= 160 * 1024, "fft_lines: line does not fit in LDS");
  TC_REQUIRE(nb != 0, "fft_lines: FFT length too large");
  auto k = nb <= 4 ? fft_lines_kernel<DIR, 4> : fft_lines_kernel<DIR, 8>;
  allow_lds((const void*)k, smem);
  hipLaunchKernelGGL(k, dim3((unsigned)m.total), dim3(1024), smem, stream, a.in,
                     a.out, F.plan(), m);
  TC_HIP(hipGetLastError());
}

bool fft_ct_enabled() {
  const char* e = std::getenv("TOMOCAM_HIP_CT_LINES");
  return !(e && e[0] == '0');
}

void fft_lines(const LineFFTArgs& a, int dir, hipStream_t stream) {
  TC_REQUIRE(a.nin + a.nin_hi <= a.L && a.nout + a.nout_hi <= a.L,
             "fft_lines: nin/nout exceed L");
  if (fft_ct_enabled() && fft_lines_ct(a, dir, stream)) return;
  if (dir < 0)
    launch_lines<-1>(a, stream);
  else
    launch_lines<1>(a, stream);
}

// ---------------------------------------------------------------------------
// real rows and rays on runtime plans (RealRowsArgs, RayArgs): a pair of rows
// or rays of one slice per line
// ---------------------------------------------------------------------------

__global__ void __launch_bounds__(RT_MAX_THREADS)
rt_r2c_rows_kernel(RealRowsArgs a, RtPlan P, int lpw) {
  extern __shared__ float2 sm[];
  const int tid = threadIdx.x, nthr = blockDim.x, L = P.L, H = L / 2 + 1;
  const int npair = (a.nm + 1) / 2, lo = (a.nm + 1) / 2, hi = a.nm / 2;
  const long g0 = (long)blockIdx.x * lpw, nlines = (long)a.nsl * npair;
  for (int q = tid; q < lpw * L; q += nthr) {
    const int l = q / L, i = q - l * L;
    const long gl = g0 + l;
    float2 w = make_float2(0.f, 0.f);
    if (gl < nlines && (i < lo || i >= L - hi)) {
      const long s = gl / npair;
      const int ka = 2 * (int)(gl - s * npair);
      const int k = i < lo ? i + hi : i - (L - hi);
      const float* f = a.real_in + (s * a.nm + ka) * a.nm;
      w.x = f[k] * a.corr[k] * a.corr[ka];
      if (ka + 1 < a.nm) w.y = f[a.nm + k] * a.corr[k] * a.corr[ka + 1];
    }
    sm[l * P.ldl + rt_pad(i)] = w;
  }
  __syncthreads();
  const float2* z = rt_fft<-1>(sm, lpw, P, tid, nthr);
  for (int q = tid; q < lpw * ((H + HG_B - 1) / HG_B * HG_B); q += nthr) {
    const int kb = q / (HG_B * lpw), l = q / HG_B - kb * lpw;
    const int k = kb * HG_B + q % HG_B;
    const long gl = g0 + l;
    if (k >= H || gl >= nlines) continue;
    const long s = gl / npair;
    const int ka = 2 * (int)(gl - s * npair);
    const float2 zk = z[l * P.ldl + rt_pad(k)];
    const float2 zm = cconj(z[l * P.ldl + rt_pad(k == 0 ? 0 : L - k)]);
    const float2 sp = cadd(zk, zm), df = csub(zk, zm);
    const int ra = ka < hi ? L + ka - hi : ka - hi;
    const int rb = ka + 1 < hi ? L + ka + 1 - hi : ka + 1 - hi;
    float2* half = a.half + s * half_grid_size(L);
    half[half_at(L, ra, k)] = make_float2(0.5f * sp.x, 0.5f * sp.y);
    if (ka + 1 < a.nm)
      half[half_at(L, rb, k)] = make_float2(0.5f * df.y, -0.5f * df.x);
  }
}

__global__ void __launch_bounds__(RT_MAX_THREADS)
rt_c2r_rows_kernel(RealRowsArgs a, RtPlan P, int lpw) {
  extern __shared__ float2 sm[];
  const int tid = threadIdx.x, nthr = blockDim.x, L = P.L, H = L / 2 + 1;
  const int npair = (a.nm + 1) / 2, hi = a.nm / 2;
  const long g0 = (long)blockIdx.x * lpw, nlines = (long)a.nsl * npair;
  for (int q = tid; q < lpw * ((H + HG_B - 1) / HG_B * HG_B); q += nthr) {
    const int kb = q / (HG_B * lpw), l = q / HG_B - kb * lpw;
    const int k = kb * HG_B + q % HG_B;
    if (k >= H) continue;
    const long gl = g0 + l;
    float2 x = make_float2(0.f, 0.f), y = x;
    if (gl < nlines) {
      const long s = gl / npair;
      const int ka = 2 * (int)(gl - s * npair);
      const int ra = ka < hi ? L + ka - hi : ka - hi;
      const int rb = ka + 1 < hi ? L + ka + 1 - hi : ka + 1 - hi;
      const float2* half = a.half + s * half_grid_size(L);
      x = half[half_at(L, ra, k)];
      if (ka + 1 < a.nm) y = half[half_at(L, rb, k)];
      if (k == 0 || 2 * k == L) x.y = y.y = 0.f;  // real by symmetry
    }
    sm[l * P.ldl + rt_pad(k)] = make_float2(x.x - y.y, x.y + y.x);
    if (k > 0 && L - k >= H)
      sm[l * P.ldl + rt_pad(L - k)] = make_float2(x.x + y.y, y.x - x.y);
  }
  __syncthreads();
  const float2* z = rt_fft<1>(sm, lpw, P, tid, nthr);
  for (int q = tid; q < lpw * a.nm; q += nthr) {
    const int l = q / a.nm, k = q - l * a.nm;
    const long gl = g0 + l;
    if (gl >= nlines) break;
    const long s = gl / npair;
    const int ka = 2 * (int)(gl - s * npair);
    const float2 v = z[l * P.ldl + rt_pad(k < hi ? L + k - hi : k - hi)];
    const float c = a.corr[k];
    float* o = a.real_out + (s * a.nm + ka) * a.nm + k;
    o[0] = v.x * c * (a.corr[ka] * a.scale);
    if (ka + 1 < a.nm) o[a.nm] = v.y * c * (a.corr[ka + 1] * a.scale);
  }
}

template <bool TO_HALF>
__global__ void __launch_bounds__(RT_MAX_THREADS)
rt_ray_kernel(RayArgs a, RtPlan P, int lpw) {
  extern __shared__ float2 sm[];
  const int tid = threadIdx.x, nthr = blockDim.x;
  const int L = P.L, N = a.N, c = N / 2;
  const int npair = (a.P + 1) / 2;
  const long g0 = (long)blockIdx.x * lpw, nlines = (long)a.nsl * npair;
  for (int t = tid; t < lpw * L; t += nthr) {
    const int l = t / L, z = t - l * L;
    const long gl = g0 + l;
    float2 v = make_float2(0.f, 0.f);
    if (z < N && gl < nlines) {
      const long s = gl / npair;
      const int p = 2 * (int)(gl - s * npair);
      const bool hasb = p + 1 < a.P;
      if constexpr (TO_HALF) {
        const float* r = a.real_in + (s * a.P + p) * N;
        v.x = r[z] - ray_level(a, r);
        if (hasb) v.y = r[N + z] - ray_level(a, r + N);
      } else {
        const float2* r = a.half_in + (s * a.P + p) * a.nh;
        v = ray_pair_sample(r, hasb ? r + a.nh : nullptr, z - c, N);
      }
      v = cmul(v, a.chirp[z]);
    }
    sm[l * P.ldl + rt_pad(z)] = v;
  }
  __syncthreads();
  float2* z = rt_fft<-1>(sm, lpw, P, tid, nthr);
  for (int t = tid; t < lpw * L; t += nthr) {
    const int l = t / L, k = t - l * L;
    float2& v = z[l * P.ldl + rt_pad(k)];
    v = cmul(v, a.bhat[k]);
  }
  __syncthreads();
  z = rt_fft<1>(sm, lpw, P, tid, nthr, z != sm);
  for (int t = tid; t < lpw * N; t += nthr) {
    const int l = t / N, j = t - l * N;
    const long gl = g0 + l;
    if (gl >= nlines) break;
    float2& y = z[l * P.ldl + rt_pad(j)];
    const float2 v = cmul(y, a.chirp[j]);
    if constexpr (TO_HALF) {
      y = v;
    } else {
      const long s = gl / npair;
      const int p = 2 * (int)(gl - s * npair);
      float* o = a.real_out + (s * a.P + p) * N + j;
      o[0] = v.x * a.scale;
      if (p + 1 < a.P) o[N] = v.y * a.scale;
    }
  }
  if constexpr (TO_HALF) {
    __syncthreads();
    for (int t = tid; t < lpw * a.nh; t += nthr) {
      const int l = t / a.nh, m = t - l * a.nh;
      if (g0 + l >= nlines) break;
      const float2* y = z + l * P.ldl;
      ray_store_pair(a, g0 + l, y[rt_pad(c + m < N ? c + m : 0)],
                     y[rt_pad(c - m)], m);
    }
  }
}

// Rows and rays too long for two LDS buffers: packed into complex lines
// z[line][L] in memory, transformed there, and taken apart.
__global__ void long_rows_pack_kernel(RealRowsArgs a, float2* z, int r2c) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int npair = (a.nm + 1) / 2, hi = a.nm / 2, lo = (a.nm + 1) / 2;
  if (idx >= (long)a.nsl * npair * a.L) return;
  const long line = idx / a.L;
  const int i = (int)(idx - line * a.L);
  const long s = line / npair;
  const int ka = 2 * (int)(line - s * npair);
  const bool hasb = ka + 1 < a.nm;
  float2 w = make_float2(0.f, 0.f);
  if (r2c) {
    if (i < lo || i >= a.L - hi) {
      const int k = i < lo ? i + hi : i - (a.L - hi);
      const float* f = a.real_in + (s * a.nm + ka) * a.nm;
      w.x = f[k] * a.corr[k] * a.corr[ka];
      if (hasb) w.y = f[a.nm + k] * a.corr[k] * a.corr[ka + 1];
    }
  } else {
    const bool low = i <= a.L / 2;
    const int k = low ? i : a.L - i;
    const int ra = ka < hi ? a.L + ka - hi : ka - hi;
    const int rb = ka + 1 < hi ? a.L + ka + 1 - hi : ka + 1 - hi;
    const float2* half = a.half + s * half_grid_size(a.L);
    float2 x = half[half_at(a.L, ra, k)];
    float2 y = hasb ? half[half_at(a.L, rb, k)] : make_float2(0.f, 0.f);
    if (k == 0 || 2 * k == a.L) x.y = y.y = 0.f;
    w = low ? make_float2(x.x - y.y, x.y + y.x)
            : make_float2(x.x + y.y, y.x - x.y);
  }
  z[idx] = w;
}

__global__ void long_rows_unpack_kernel(RealRowsArgs a, const float2* z,
                                        int r2c) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int npair = (a.nm + 1) / 2, hi = a.nm / 2;
  const int width = r2c ? a.L / 2 + 1 : a.nm;
  if (idx >= (long)a.nsl * npair * width) return;
  const long line = idx / width;
  const int k = (int)(idx - line * width);
  const long s = line / npair;
  const int ka = 2 * (int)(line - s * npair);
  const bool hasb = ka + 1 < a.nm;
  z += line * a.L;
  if (r2c) {
    const float2 zk = z[k], zm = cconj(z[k == 0 ? 0 : a.L - k]);
    const float2 sp = cadd(zk, zm), df = csub(zk, zm);
    const int ra = ka < hi ? a.L + ka - hi : ka - hi;
    const int rb = ka + 1 < hi ? a.L + ka + 1 - hi : ka + 1 - hi;
    float2* half = a.half + s * half_grid_size(a.L);
    half[half_at(a.L, ra, k)] = make_float2(0.5f * sp.x, 0.5f * sp.y);
    if (hasb)
      half[half_at(a.L, rb, k)] = make_float2(0.5f * df.y, -0.5f * df.x);
  } else {
    const float2 v = z[k < hi ? a.L + k - hi : k - hi];
    const float c = a.corr[k];
    float* o = a.real_out + (s * a.nm + ka) * a.nm + k;
    o[0] = v.x * c * (a.corr[ka] * a.scale);
    if (hasb) o[a.nm] = v.y * c * (a.corr[ka + 1] * a.scale);
  }
}

__global__ void long_rays_pack_kernel(RayArgs a, float2* z, int to_half) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int npair = (a.P + 1) / 2, c = a.N / 2;
  if (idx >= (long)a.nsl * npair * a.L) return;
  const long line = idx / a.L;
  const int i = (int)(idx - line * a.L);
  const long s = line / npair;
  const int p = 2 * (int)(line - s * npair);
  const bool hasb = p + 1 < a.P;
  float2 v = make_float2(0.f, 0.f);
  if (i < a.N) {
    if (to_half) {
      const float* r = a.real_in + (s * a.P + p) * a.N;
      v.x = r[i] - ray_level(a, r);
      if (hasb) v.y = r[a.N + i] - ray_level(a, r + a.N);
    } else {
      const float2* r = a.half_in + (s * a.P + p) * a.nh;
      v = ray_pair_sample(r, hasb ? r + a.nh : nullptr, i - c, a.N);
    }
    v = cmul(v, a.chirp[i]);
  }
  z[idx] = v;
}

__global__ void long_rays_mul_kernel(float2* z, const float2* bhat, int L,
                                     long n) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx < n) z[idx] = cmul(z[idx], bhat[idx % L]);
}

__global__ void long_rays_unpack_kernel(RayArgs a, const float2* z,
                                        int to_half) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int npair = (a.P + 1) / 2, c = a.N / 2;
  const int width = to_half ? a.nh : a.N;
  if (idx >= (long)a.nsl * npair * width) return;
  const long line = idx / width;
  const int j = (int)(idx - line * width);
  z += line * a.L;
  if (to_half) {
    const int jp = c + j < a.N ? c + j : 0, jn = c - j;
    ray_store_pair(a, line, cmul(z[jp], a.chirp[jp]), cmul(z[jn], a.chirp[jn]),
                   j);
  } else {
    const long s = line / npair;
    const int p = 2 * (int)(line - s * npair);
    const float2 v = cmul(z[j], a.chirp[j]);
    float* o = a.real_out + (s * a.P + p) * a.N + j;
    o[0] = v.x * a.scale;
    if (p + 1 < a.P) o[a.N] = v.y * a.scale;
  }
}

static void long_lines(float2* z, int L, long nlines, int dir,
                       hipStream_t stream) {
  LineFFTArgs l;
  l.in = l.out = z;
  l.L = l.nin = l.nout = L;
  l.lines_per_batch = (int)nlines;
  l.lstride = L;
  fft_lines(l, dir, stream);
}

static void long_rows(RealRowsArgs a, bool r2c, hipStream_t stream) {
  const int nsl = a.nsl, npair = (a.nm + 1) / 2;
  DevBuf z(sizeof(float2) * (size_t)npair * a.L);
  a.nsl = 1;  // a slice at a time: the lines take as much room as its half grid
  for (int s = 0; s < nsl; ++s) {
    hipLaunchKernelGGL(long_rows_pack_kernel,
                       dim3(cdiv((size_t)npair * a.L, 256)), dim3(256), 0,
                       stream, a, z.as<float2>(), r2c ? 1 : 0);
    TC_HIP(hipGetLastError());
    long_lines(z.as<float2>(), a.L, npair, r2c ? -1 : 1, stream);
    const size_t n = (size_t)npair * (r2c ? a.L / 2 + 1 : a.nm);
    hipLaunchKernelGGL(long_rows_unpack_kernel, dim3(cdiv(n, 256)), dim3(256),
                       0, stream, a, z.as<float2>(), r2c ? 1 : 0);
    TC_HIP(hipGetLastError());
    if (r2c) a.real_in += (long)a.nm * a.nm;
    else a.real_out += (long)a.nm * a.nm;
    a.half += half_grid_size(a.L);
  }
}

static void long_rays(RayArgs a, bool to_half, hipStream_t stream) {
  const int nsl = a.nsl, npair = (a.P + 1) / 2;
  const size_t nz = (size_t)npair * a.L;
  DevBuf z(sizeof(float2) * nz);
  a.nsl = 1;
  for (int s = 0; s < nsl; ++s) {
    hipLaunchKernelGGL(long_rays_pack_kernel, dim3(cdiv(nz, 256)), dim3(256), 0,
                       stream, a, z.as<float2>(), to_half ? 1 : 0);
    TC_HIP(hipGetLastError());
    long_lines(z.as<float2>(), a.L, npair, -1, stream);
    hipLaunchKernelGGL(long_rays_mul_kernel, dim3(cdiv(nz, 256)), dim3(256), 0,
                       stream, z.as<float2>(), a.bhat, a.L, (long)nz);
    TC_HIP(hipGetLastError());
    long_lines(z.as<float2>(), a.L, npair, 1, stream);
    const size_t n = (size_t)npair * (to_half ? a.nh : a.N);
    hipLaunchKernelGGL(long_rays_unpack_kernel, dim3(cdiv(n, 256)), dim3(256),
                       0, stream, a, z.as<float2>(), to_half ? 1 : 0);
    TC_HIP(hipGetLastError());
    if (to_half) {
      a.real_in += (long)a.P * a.N;
      a.half_out += (long)a.P * a.nh;
    } else {
      a.half_in += (long)a.P * a.nh;
      a.real_out += (long)a.P * a.N;
    }
  }
}

void fft_real_rows(const RealRowsArgs& a, bool r2c, hipStream_t stream) {
  TC_REQUIRE(a.nm >= 1 && a.nm <= a.L && a.L % 2 == 0,
             "fft_real_rows: bad shape");
  if (fft_ct_enabled() && fft_real_rows_ct(a, r2c, stream)) return;
  const long nlines = (long)a.nsl * ((a.nm + 1) / 2);
  if (nlines == 0) return;
  if (!rt_fits(a.L)) return long_rows(a, r2c, stream);
  const RtLaunch l = rt_launch(a.L, nlines, 4);
  auto k = r2c ? rt_r2c_rows_kernel : rt_c2r_rows_kernel;
  allow_lds((const void*)k, l.smem);
  hipLaunchKernelGGL(k, dim3(cdiv(nlines, l.lpw)), dim3(l.nthr), l.smem, stream,
                     a, l.plan, l.lpw);
  TC_HIP(hipGetLastError());
}

void fft_rays(const RayArgs& a, bool to_half, hipStream_t stream) {
  const long nlines = (long)a.nsl * ((a.P + 1) / 2);
  if (nlines <= 0) return;
  if (fft_ct_enabled() && fft_rays_ct(a, to_half, stream)) return;
  TC_REQUIRE(2 * a.N - 1 <= a.L, "ray DFT: length too short");
  if (!rt_fits(a.L)) return long_rays(a, to_half, stream);
  const RtLaunch l = rt_launch(a.L, nlines, 4);
  auto k = to_half ? rt_ray_kernel<true> : rt_ray_kernel<false>;
  allow_lds((const void*)k, l.smem);
  hipLaunchKernelGGL(k, dim3(cdiv(nlines, l.lpw)), dim3(l.nthr), l.smem, stream,
                     a, l.plan, l.lpw);
  TC_HIP(hipGetLastError());
}

// Column transforms restricted to the columns [0, lo) and [cols - hi, cols)
// (the others are not needed, or are zero, in the caller).
static void fft_cols_ranges(float2* data, int nbatch, int rows, int cols,
                            long row_pitch, long slice_pitch, int lo, int hi,
                            int dir, hipStream_t stream) {
  if (lo + hi >= cols) {
    lo = cols;
    hi = 0;
  }
  LineFFTArgs a;
  a.L = rows;
  a.nbatch = nbatch;
  a.bstride = slice_pitch;
  a.lstride = 1;
  a.estride = row_pitch;
  a.nin = rows;
  a.nout = rows;
  a.colmajor = true;
  if (lo > 0) {
    a.in = a.out = data;
    a.lines_per_batch = lo;
    fft_lines(a, dir, stream);
  }
  if (hi > 0) {
    a.in = a.out = data + (cols - hi);
    a.lines_per_batch = hi;
    fft_lines(a, dir, stream);
  }
}

static void fft_rows_all(float2* data, int nbatch, int rows, int cols,
                         long row_pitch, long slice_pitch, int dir,
                         hipStream_t stream) {
  LineFFTArgs a;
  a.in = data;
  a.out = data;
  a.L = cols;
  a.lines_per_batch = rows;
  a.nbatch = nbatch;
  a.bstride = slice_pitch;
  a.lstride = row_pitch;
  a.estride = 1;
  a.nin = cols;
  a.nout = cols;
  a.colmajor = false;
  fft_lines(a, dir, stream);
}

void fft2d_pruned(float2* data, int nbatch, int n, int lo, int hi, int dir,
                  bool rows_first, hipStream_t stream) {
  const long pitch = n, slice = (long)n * n;
  if (rows_first) {
    fft_rows_all(data, nbatch, n, n, pitch, slice, dir, stream);
    fft_cols_ranges(data, nbatch, n, n, pitch, slice, lo, hi, dir, stream);
  } else {
    fft_cols_ranges(data, nbatch, n, n, pitch, slice, lo, hi, dir, stream);
    fft_rows_all(data, nbatch, n, n, pitch, slice, dir, stream);
  }
}

void fft2d(float2* data, int nbatch, int rows, int cols, long row_pitch,
           long slice_pitch, int dir, hipStream_t stream) {
  LineFFTArgs a;
  // rows: contiguous lines
  a.in = data;
  a.out = data;
  a.L = cols;
  a.lines_per_batch = rows;
  a.nbatch = nbatch;
  a.bstride = slice_pitch;
  a.lstride = row_pitch;
  a.estride = 1;
  a.nin = cols;
  a.nout = cols;
  a.colmajor = false;
  fft_lines(a, dir, stream);
  // columns
  a.L = rows;
  a.lines_per_batch = cols;
  a.lstride = 1;
  a.estride = row_pitch;
  a.nin = rows;
  a.nout = rows;
  a.colmajor = true;
  fft_lines(a, dir, stream);
}

}  // namespace tc
