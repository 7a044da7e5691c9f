// Toeplitz normal operator: PSF spectrum set-up and the three-pass apply.
// Reference: src/toeplitz.h:51-159 (PointSpreadFunction ctor / convolve).
#include <hip/hip_fp16.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <initializer_list>
#include <map>
#include <mutex>
#include <utility>
#include <vector>

#include "fft_device.h"
#include "fft_ops.h"
#include "lds_launch.h"
#include "toeplitz.h"

namespace tc {

// lines per workgroup of the compile-time plan for FFT length M (0: none)
int toeplitz_ct_lpw(int M);
extern const int kToeplitzCtSizes[];
extern const float kToeplitzCtCost[];
extern const int kToeplitzCtCount;
int toeplitz_plan_length(int m, int most);
bool toeplitz_ct_prepare(int M);

// Compile-time plan sizes eligible for an n x n Toeplitz product: >= 2n - 1
// and within 10 % of the smallest even 2,3,5,7-smooth length, ordered by
// size x measured relative cost per point (cheapest first).
static std::vector<int> toeplitz_ct_candidates(int n) {
  const int m = 2 * n - 1;
  const int smooth = fft_next_smooth(m, true);
  std::vector<std::pair<float, int>> c;
  for (int i = 0; i < kToeplitzCtCount; ++i) {
    const int L = kToeplitzCtSizes[i];
    if (L < m || L > smooth + smooth / 10) continue;
    c.emplace_back((float)L * kToeplitzCtCost[i], L);
  }
  std::stable_sort(c.begin(), c.end(),
                   [](const std::pair<float, int>& a,
                      const std::pair<float, int>& b) {
                     return a.first < b.first;
                   });
  std::vector<int> out;
  for (auto& x : c) out.push_back(x.second);
  return out;
}

// FFT lengths picked by Psf::tune_length, keyed by (device, n)
static std::mutex g_len_mu;
static std::map<std::pair<int, int>, int> g_len_tuned;

static std::pair<int, int> len_key(int n) {
  int dev = 0;
  TC_HIP(hipGetDevice(&dev));
  return std::make_pair(dev, n);
}

// FFT length for an n x n Toeplitz product: any even length >= 2n - 1 gives
// the same result.  The autotuner's choice for this width if there is one;
// else among the eligible compile-time plan sizes the one with the least
// size x relative cost per point (they come first because they alone have the
// mixed-precision forms, and an operator serves both); with none, from 486 on
// the cheapest plan of any kind within 1/7 of the smallest even smooth length,
// which every width from 243 to 4096 has (there without the mixed forms, see
// has_mixed), else that length.  Runtime-plan kernels against the plan: 2 x 849^2
// 98 and 54 us; 4 x 330^2, 672 and 768 points, 35 and 27 us; 2 x 1310^2, 2646
// and 2916, 280 and 72 us; 2 x 2620^2, 5250 and 5832, 1003 and 293 us; 2 x
// 3000^2, 6000 and 6144, 1279 and 425 us.  Shorter lengths have no plans: trial
// ones took 13.5 instead of 18.8 us at 1 x 128^2 and 21.1 instead of 23.9 at 1
// x 181^2.
int toeplitz_fft_length(int n) {
  {
    // (no device query while nothing is tuned: the rule works without one)
    std::lock_guard<std::mutex> lk(g_len_mu);
    if (!g_len_tuned.empty()) {
      auto it = g_len_tuned.find(len_key(n));
      if (it != g_len_tuned.end()) return it->second;
    }
  }
  const std::vector<int> c = toeplitz_ct_candidates(n);
  if (!c.empty()) return c[0];
  const int smooth = fft_next_smooth(2 * n - 1, true);
  const int plan = smooth < 486
                       ? 0
                       : toeplitz_plan_length(2 * n - 1, smooth + smooth / 7);
  return plan > 0 ? plan : smooth;
}

// ---------------------------------------------------------------------------
// PSF spectrum
// ---------------------------------------------------------------------------

// C[i2][i1] = PSF(m1, m2) with m = i (i < n) or i - M (i > M - n), else 0.
__global__ void psf_place_kernel(const float* __restrict__ psf, float2* c,
                                 int n, int M) {
  long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (long)M * M) return;
  int i2 = (int)(idx / M);
  int i1 = (int)(idx - (long)i2 * M);
  int m1 = i1 < n ? i1 : (i1 > M - n ? i1 - M : M);
  int m2 = i2 < n ? i2 : (i2 > M - n ? i2 - M : M);
  float v = 0.f;
  if (m1 != M && m2 != M) {
    const int n1 = 2 * n - 1;
    v = psf[(long)(m2 + n - 1) * n1 + (m1 + n - 1)];
  }
  c[idx] = make_float2(v, 0.f);
}

// spec[k1][k2] = Re C[k2][k1] * scale, k1 < H, k2 < M
__global__ void psf_extract_kernel(const float2* __restrict__ c, float* spec,
                                   int M, int H, float scale) {
  long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (long)M * H) return;
  int k1 = (int)(idx / M);
  int k2 = (int)(idx - (long)k1 * M);
  spec[idx] = c[(long)k2 * M + k1].x * scale;
}

Psf::Psf(const float* d_psf, int n, hipStream_t stream) : n_(n) {
  TC_REQUIRE(n >= 2, "PSF: image width must be >= 2");
  rp_ = n + (n & 1);  // rows of the workspace: whole pairs
  const size_t n1 = 2 * (size_t)n - 1;
  arr_.alloc(sizeof(float) * n1 * n1);
  TC_HIP(hipMemcpyAsync(arr_.as<void>(), d_psf, sizeof(float) * n1 * n1,
                        hipMemcpyDeviceToDevice, stream));
  build_spectrum(toeplitz_fft_length(n), stream);
}

void Psf::build_spectrum(int M, hipStream_t stream) {
  M_ = M;
  H_ = M_ / 2 + 1;
  // the mixed forms serve the widths whose smooth length is within 10 %
  const std::vector<int> c10 = toeplitz_ct_candidates(n_);
  mixed_ = std::find(c10.begin(), c10.end(), M_) != c10.end();
  {
    ArenaPause no_arena;  // process-lifetime tables
    if (!toeplitz_ct_prepare(M_)) fft_length(M_);
  }
  // everything sized by the FFT length starts over
  spec16_.release();
  spec16_exp_ = 0;
  cinv_.release();
  cinv_slices_ = 0;
  work_.release();
  work_slices_ = 0;
  DevBuf c(sizeof(float2) * (size_t)M_ * M_);
  long tot = (long)M_ * M_;
  hipLaunchKernelGGL(psf_place_kernel, dim3(cdiv(tot, 256)), dim3(256), 0,
                     stream, arr_.as<float>(), c.as<float2>(), n_, M_);
  TC_HIP(hipGetLastError());
  // the spectrum keeps columns k1 < H only (real, even PSF)
  fft2d_pruned(c.as<float2>(), 1, M_, H_, 0, -1, true, stream);
  spec_.alloc(sizeof(float) * (size_t)M_ * H_);
  const double scale = 1.0 / ((double)n_ * n_ * n_ * (double)M_ * M_);
  long tot2 = (long)M_ * H_;
  hipLaunchKernelGGL(psf_extract_kernel, dim3(cdiv(tot2, 256)), dim3(256), 0,
                     stream, c.as<float2>(), spec_.as<float>(), M_, H_,
                     (float)scale);
  TC_HIP(hipGetLastError());
  TC_HIP(hipStreamSynchronize(stream));
}

int Psf::tune_length(int nslices, hipStream_t stream) {
  const std::vector<int> cands = toeplitz_ct_candidates(n_);
  if (cands.size() < 2) return 0;
  {
    std::lock_guard<std::mutex> lk(g_len_mu);
    auto it = g_len_tuned.find(len_key(n_));
    if (it != g_len_tuned.end()) {
      if (it->second != M_) build_spectrum(it->second, stream);
      return -1;
    }
  }
  // one application of each candidate length on scratch data (one stream,
  // the 144 MB rule's groups), best of two timed runs after a warm-up; the
  // static rule's choice (first) is replaced only by one >= 5 % faster: the
  // length changes T x in the last bits, so near-ties stay on the rule and
  // results stay the same from process to process
  constexpr float kMargin = 0.05f;
  const int S = std::max(1, nslices);
  const long tot = (long)n_ * n_ * S;
  DevBuf x(sizeof(float) * (size_t)tot), out(sizeof(float) * (size_t)tot);
  TC_HIP(hipMemsetAsync(x.as<void>(), 0, sizeof(float) * (size_t)tot, stream));
  hipEvent_t e0, e1;
  TC_HIP(hipEventCreate(&e0));
  TC_HIP(hipEventCreate(&e1));
  int best = 0;
  float best_ms = 0.f;
  try {
    for (int L : cands) {
      if (L != M_) build_spectrum(L, stream);
      float ms = 0.f;
      for (int rep = 0; rep < 3; ++rep) {
        TC_HIP(hipEventRecord(e0, stream));
        apply(x.as<float>(), nullptr, out.as<float>(), S, 0, nullptr, stream);
        TC_HIP(hipEventRecord(e1, stream));
        TC_HIP(hipEventSynchronize(e1));
        float t = 0.f;
        TC_HIP(hipEventElapsedTime(&t, e0, e1));
        if (rep == 1 || (rep > 1 && t < ms)) ms = t;
      }
      if (tune_log())
        std::fprintf(stderr,
                     "[tomocam] toeplitz tune n=%d, %d slices: length %d: "
                     "%.3f ms\n", n_, S, L, (double)ms);
      if (best == 0 || ms < (1.0f - kMargin) * best_ms) {
        best = L;
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
  {
    std::lock_guard<std::mutex> lk(g_len_mu);
    g_len_tuned[len_key(n_)] = best;
  }
  if (best != M_) build_spectrum(best, stream);
  return best;
}

void Psf::reserve(int nslices) {
  if ((size_t)nslices > work_slices_) {
    work_.alloc(sizeof(float2) * (size_t)nslices * H_ * rp_);
    work_slices_ = nslices;
  }
}

// ---------------------------------------------------------------------------
// pass A: pair-packed forward row FFTs -> Wt[s][k1][row]
// ---------------------------------------------------------------------------

template <int NB>
__global__ void __launch_bounds__(1024)
toep_rows_fwd(const float* __restrict__ x, float2* __restrict__ wt, FFTPlan P,
              int n, int H, int rp, int lpw, int nbps) {
  extern __shared__ float2 sm[];
  const int tid = threadIdx.x, nthr = blockDim.x;
  const int M = P.L;
  const int b = xcd_remap(blockIdx.x, gridDim.x);
  const int s = b / nbps;
  const int r0 = (b - s * nbps) * 2 * lpw;
  const float* xs = x + (long)s * n * n;
  for (int t = tid; t < lpw * M; t += nthr) {
    int l = t / M;
    int c = t - l * M;
    int ra = r0 + 2 * l;
    float re = 0.f, im = 0.f;
    if (c < n) {
      if (ra < n) re = xs[(long)ra * n + c];
      if (ra + 1 < n) im = xs[(long)(ra + 1) * n + c];
    }
    sm[t] = make_float2(re, im);
  }
  __syncthreads();
  fft_lds<-1, NB>(sm, lpw, M, P, tid, nthr);
  float2* ws = wt + (long)s * H * rp;
  for (int t = tid; t < lpw * H; t += nthr) {
    int k = t / lpw;
    int l = t - k * lpw;
    int ra = r0 + 2 * l;
    if (ra < rp) {
      float2 zk = sm[l * M + k];
      float2 zm = cconj(sm[l * M + (k == 0 ? 0 : M - k)]);
      float2 sp = cadd(zk, zm), df = csub(zk, zm);
      float4 q = make_float4(0.5f * sp.x, 0.5f * sp.y, 0.5f * df.y,
                             -0.5f * df.x);
      *reinterpret_cast<float4*>(ws + (long)k * rp + ra) = q;
    }
  }
}

// ---------------------------------------------------------------------------
// pass B: column FFT, multiply by the real spectrum, inverse column FFT
// ---------------------------------------------------------------------------

template <int NB>
__global__ void __launch_bounds__(1024)
toep_cols(float2* __restrict__ wt, const float* __restrict__ spec, FFTPlan P,
          int n, int H, int rp, int lpw, int nbps, double* partials) {
  extern __shared__ float2 sm[];
  __shared__ double red[16];
  const int tid = threadIdx.x, nthr = blockDim.x;
  const int M = P.L;
  const int b = xcd_remap(blockIdx.x, gridDim.x);
  const int s = b / nbps;
  const int k0 = (b - s * nbps) * lpw;
  float2* ws = wt + (long)s * H * rp;
  for (int t = tid; t < lpw * M; t += nthr) {
    int l = t / M;
    int r = t - l * M;
    float2 v = make_float2(0.f, 0.f);
    if (r < n && k0 + l < H) v = ws[(long)(k0 + l) * rp + r];
    sm[t] = v;
  }
  __syncthreads();
  fft_lds<-1, NB>(sm, lpw, M, P, tid, nthr);
  double acc = 0.0;
  for (int t = tid; t < lpw * M; t += nthr) {
    int l = t / M;
    int k2 = t - l * M;
    int k1 = k0 + l;
    if (k1 < H) {
      float h = spec[(long)k1 * M + k2];
      float2 v = sm[t];
      float wgt = (k1 == 0 || 2 * k1 == M) ? 1.f : 2.f;
      acc += (double)(wgt * h * (v.x * v.x + v.y * v.y));
      sm[t] = cscale(v, h);
    }
  }
  __syncthreads();
  fft_lds<1, NB>(sm, lpw, M, P, tid, nthr);
  for (int t = tid; t < lpw * M; t += nthr) {
    int l = t / M;
    int r = t - l * M;
    if (r < n && k0 + l < H) ws[(long)(k0 + l) * rp + r] = sm[t];
  }
  if (partials) {
    double tot = block_sum(acc, red);
    if (tid == 0) partials[b] = tot;
  }
}

// ---------------------------------------------------------------------------
// pass C: pair-packed inverse row FFTs, crop, epilogue
// ---------------------------------------------------------------------------

template <int NB, int MODE>
__global__ void __launch_bounds__(1024)
toep_rows_inv(const float2* __restrict__ wt, const float* __restrict__ bvec,
              float* __restrict__ out, FFTPlan P, int n, int H, int rp,
              int lpw, int nbps) {
  extern __shared__ float2 sm[];
  const int tid = threadIdx.x, nthr = blockDim.x;
  const int M = P.L;
  const int b = xcd_remap(blockIdx.x, gridDim.x);
  const int s = b / nbps;
  const int r0 = (b - s * nbps) * 2 * lpw;
  const float2* ws = wt + (long)s * H * rp;
  for (int t = tid; t < lpw * H; t += nthr) {
    int k = t / lpw;
    int l = t - k * lpw;
    int ra = r0 + 2 * l;
    float4 q = make_float4(0.f, 0.f, 0.f, 0.f);
    if (ra < rp) q = *reinterpret_cast<const float4*>(ws + (long)k * rp + ra);
    if (k == 0 || 2 * k == M) {
      q.y = 0.f;
      q.w = 0.f;
    }
    // z = X1 + i X2
    sm[l * M + k] = make_float2(q.x - q.w, q.y + q.z);
    if (k > 0 && M - k >= H) {
      // z[M-k] = conj(X1) + i conj(X2)
      sm[l * M + M - k] = make_float2(q.x + q.w, q.z - q.y);
    }
  }
  __syncthreads();
  fft_lds<1, NB>(sm, lpw, M, P, tid, nthr);
  const long so = (long)s * n * n;
  for (int t = tid; t < lpw * n; t += nthr) {
    int l = t / n;
    int c = t - l * n;
    int ra = r0 + 2 * l;
    float2 v = sm[l * M + c];
    if (ra < n) {
      long o = so + (long)ra * n + c;
      out[o] = MODE == 1 ? v.x - bvec[o] : v.x;
    }
    if (ra + 1 < n) {
      long o = so + (long)(ra + 1) * n + c;
      out[o] = MODE == 1 ? v.y - bvec[o] : v.y;
    }
  }
}

// ---------------------------------------------------------------------------

__global__ void reduce_partials_kernel(const double* __restrict__ p, long n,
                                       double* out) {
  __shared__ double red[16];
  double acc = 0.0;
  for (long i = threadIdx.x; i < n; i += blockDim.x) acc += p[i];
  double tot = block_sum(acc, red);
  if (threadIdx.x == 0) out[0] = tot;
}

void reduce_partials(const double* partials, long n, double* out,
                     hipStream_t stream) {
  hipLaunchKernelGGL(reduce_partials_kernel, dim3(1), dim3(1024), 0, stream,
                     partials, n, out);
  TC_HIP(hipGetLastError());
}

bool toeplitz_apply_ct(int M, const float* x, const float* b, float* out,
                       float2* wt, const float* spec, int n, int H, int rp,
                       int nslices, int mode, double* partials,
                       hipStream_t stream, double img_b, double spec_b,
                       const Psf::StepCommit* cm, const ToeplitzStreams* ts,
                       int group_cap = 0);
int toeplitz_streams(int H, int rp, int elem_bytes, int nslices);
int toeplitz_rule_group(int nslices, int H, int rp, int elem_bytes);
void toeplitz_set_streams(int H, int rp, int elem_bytes, int nslices,
                          int streams);

Psf::~Psf() {
  for (int k = 0; k < kMaxToeplitzStreams - 1; ++k) {
    if (ts_.aux[k]) (void)hipStreamDestroy(ts_.aux[k]);
    if (ts_.done[k]) (void)hipEventDestroy(ts_.done[k]);
  }
  if (ts_.start) (void)hipEventDestroy(ts_.start);
}

bool Psf::single_stream(int nslices, bool half) const {
  return toeplitz_streams(H_, rp_, half ? 4 : 8, nslices) < 2;
}

const ToeplitzStreams* Psf::streams_for(int nslices, int elem_bytes) {
  const int st = toeplitz_streams(H_, rp_, elem_bytes, nslices);
  if (st < 2) return nullptr;
  if (!ts_.start)
    TC_HIP(hipEventCreateWithFlags(&ts_.start, hipEventDisableTiming));
  for (int k = 0; k < st - 1; ++k)
    if (!ts_.aux[k]) {
      // default priority, non-blocking: ordered only by the events
      TC_HIP(hipStreamCreateWithFlags(&ts_.aux[k], hipStreamNonBlocking));
      TC_HIP(hipEventCreateWithFlags(&ts_.done[k], hipEventDisableTiming));
    }
  ts_.n = st;
  return &ts_;
}

// spec: the FP16 copy with FP16 intermediates (wt16), else the FP32 one
bool toeplitz_apply_ct_half(int M, const void* x16, float* out, void* wt,
                            const void* spec, int n, int H, int rp,
                            int nslices, double* partials, hipStream_t stream,
                            double img_b, double spec_b,
                            const Psf::StepCommit* sc,
                            const ToeplitzHalf& half, bool wt16,
                            const ToeplitzStreams* ts);
int toeplitz_half_group(int nslices, int H, int rp);
int toeplitz_ct_scales(int M, int H);

// max |v[i]| over n floats into out[0] (one workgroup)
__global__ void absmax_kernel(const float* __restrict__ v, long n,
                              float* out) {
  __shared__ float red[16];
  float m = 0.f;
  for (long i = threadIdx.x; i < n; i += blockDim.x) m = fmaxf(m, fabsf(v[i]));
  for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w) m = fmaxf(m, red[w]);
    out[0] = m;
  }
}

__global__ void to_half_kernel(const float* __restrict__ v, __half* out,
                               long n, float scale) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = __float2half_rn(v[i] * scale);
}

bool Psf::run_half(const void* g16, const float* gsc, float* out,
                   int nslices, double* dot_partials, const StepCommit* c,
                   hipStream_t stream, bool wt16) {
  TC_REQUIRE(nslices >= 1, "Toeplitz: need at least one slice");
  TC_REQUIRE(g16 && gsc, "Toeplitz: null FP16 input or scales");
  if (!has_mixed()) return false;
  const long nspec = (long)M_ * H_;
  // FP32 intermediates read the FP32 spectrum (an FP16 copy measured no
  // faster there, and its rounding accumulated in the MBIR's T sol
  // recurrence); FP16 intermediates read the FP16 copy
  if (wt16 && spec16_.bytes() == 0) {
    // FP16 copy of the spectrum, its largest magnitude mapped into
    // (2^13, 2^14]
    DevBuf mx(sizeof(float));
    hipLaunchKernelGGL(absmax_kernel, dim3(1), dim3(1024), 0, stream,
                       spectrum(), nspec, mx.as<float>());
    TC_HIP(hipGetLastError());
    float m = 0.f;
    TC_HIP(hipMemcpyAsync(&m, mx.as<float>(), sizeof(float),
                          hipMemcpyDeviceToHost, stream));
    TC_HIP(hipStreamSynchronize(stream));
    TC_REQUIRE(m > 0.f && std::isfinite(m), "Toeplitz: degenerate spectrum");
    int ex = 0;
    (void)std::frexp(m, &ex);
    spec16_exp_ = 14 - ex;
    spec16_.alloc(sizeof(__half) * (size_t)nspec);
    hipLaunchKernelGGL(to_half_kernel, dim3(cdiv(nspec, 256)), dim3(256), 0,
                       stream, spectrum(), spec16_.as<__half>(), nspec,
                       std::ldexp(1.0f, spec16_exp_));
    TC_HIP(hipGetLastError());
  }
  reserve(nslices);
  // pass B's output scales for one group in flight per stream
  const int group = kMaxToeplitzStreams * toeplitz_half_group(nslices, H_, rp_);
  if (wt16 && (size_t)group > cinv_slices_) {
    cinv_.alloc(sizeof(float) * (size_t)group * toeplitz_ct_scales(M_, H_));
    cinv_slices_ = group;
  }
  int nb = 0;
  (void)std::frexp((double)n_, &nb);  // 2^(nb-1) <= n < 2^nb
  ToeplitzHalf h;
  h.gsc = gsc;
  const int e = wt16 ? spec16_exp_ : 0;  // the spectrum's scale exponent
  h.sinv = std::ldexp(1.0f, -e);
  h.cinv = cinv_.as<float>();
  h.wsc = std::ldexp(1.0f, -(nb + 1));  // n * 2^16 * wsc < 2^15
  h.cbase = std::ldexp(1.0f, nb + 1 - e);
  h.pconst = wt16 ? std::ldexp(1.0f, 2 * (nb + 1) - e) : 1.0f;
  const double img_b = 4.0 * nslices * (double)n_ * n_;
  const double spec_b = 8.0 * nslices * (double)n_ * H_;
  const void* spec = wt16 ? spec16_.as<void>()
                          : static_cast<const void*>(spectrum());
  return toeplitz_apply_ct_half(M_, g16, c ? c->Tdst : out, work_.as<void>(),
                                spec, n_, H_, rp_, nslices,
                                dot_partials, stream, img_b, spec_b, c, h,
                                wt16, streams_for(nslices, wt16 ? 4 : 8));
}

bool Psf::has_fused() const { return toeplitz_ct_lpw(M_) > 0; }
bool Psf::has_mixed() const { return mixed_; }

void toeplitz_set_group(int H, int rp, int elem_bytes, int nslices,
                        int group);
bool toeplitz_group_tuned(int H, int rp, int elem_bytes, int nslices);

__global__ void fill_float_kernel(float* p, long n, float v) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

int Psf::tune_groups(int nslices, bool half, hipStream_t stream) {
  if (!(half ? has_mixed() : has_fused()) || nslices < 2) return 0;
  const int eb = half ? 4 : 8;
  if (toeplitz_group_tuned(H_, rp_, eb, nslices)) return -1;
  const long plane = (long)n_ * n_;
  const long tot = plane * nslices;
  // scratch operands: the passes' time does not depend on the values
  DevBuf x(sizeof(float) * (size_t)tot), out(sizeof(float) * (size_t)tot);
  DevBuf gsc;
  TC_HIP(hipMemsetAsync(x.as<void>(), 0, sizeof(float) * (size_t)tot, stream));
  if (half) {
    gsc.alloc(sizeof(float) * (size_t)nslices);
    hipLaunchKernelGGL(fill_float_kernel, dim3(cdiv(nslices, 256)), dim3(256),
                       0, stream, gsc.as<float>(), (long)nslices, 1.0f);
    TC_HIP(hipGetLastError());
  }
  // candidates: groups around the 144 MB rule's group r (r, r/2, 2r, capped
  // at nslices) on one stream, and r/2 and r on two streams (groups
  // alternate between the caller's stream and a second one, so one group's
  // latency-bound row passes overlap the next group's VALU-bound column
  // pass: 2.5-3 % faster at 64 x 2908^2).  The application is timed on the
  // caller's stream, which waits for the second one.
  // Candidates in order of preference; a later one replaces the best so
  // far only when at least kMargin faster, so near-ties resolve the same
  // way on every run and the configuration is reproducible.  On two streams
  // the smaller group comes first: the loop's applications (with the step
  // commit and dot partials in the last pass) overlap better in small
  // groups than this scratch application shows.  At 64 x 2908^2 one slice
  // on two streams timed 0.5 % faster here than two slices, and the
  // 100-iteration loop ran 3 % faster with it (34.4 against 33.5 slices/s).
  constexpr float kMargin = 0.02f;
  const int r = toeplitz_rule_group(nslices, H_, rp_, eb);
  std::vector<std::pair<int, int>> cands;
  for (int st : {1, 2})
    for (int g : st == 1 ? std::initializer_list<int>{r, std::max(1, r / 2),
                                                      std::min(2 * r, nslices)}
                         : std::initializer_list<int>{std::max(1, r / 2), r}) {
      if (st == 2 && (g > r || 2 * g > nslices)) continue;
      bool seen = false;
      for (auto& c : cands) seen |= c.first == g && c.second == st;
      if (!seen) cands.emplace_back(g, st);
    }
  hipEvent_t e0, e1;
  TC_HIP(hipEventCreate(&e0));
  TC_HIP(hipEventCreate(&e1));
  int best = 0, best_st = 1;
  float best_ms = 0.f;
  try {
    for (auto [g, st] : cands) {
      toeplitz_set_group(H_, rp_, eb, nslices, g);
      toeplitz_set_streams(H_, rp_, eb, nslices, st);
      float ms = 0.f;
      for (int rep = 0; rep < 3; ++rep) {  // first run warms caches
        TC_HIP(hipEventRecord(e0, stream));
        if (half)
          apply_half(x.as<void>(), gsc.as<float>(), out.as<float>(), nslices,
                     nullptr, stream);
        else
          apply(x.as<float>(), nullptr, out.as<float>(), nslices, 0, nullptr,
                stream);
        TC_HIP(hipEventRecord(e1, stream));
        TC_HIP(hipEventSynchronize(e1));
        float t = 0.f;
        TC_HIP(hipEventElapsedTime(&t, e0, e1));
        if (rep == 1 || (rep > 1 && t < ms)) ms = t;
      }
      if (tune_log())
        std::fprintf(stderr,
                     "[tomocam] toeplitz tune n=%d, %d slices: group %d, "
                     "%d stream(s): %.3f ms\n", n_, nslices, g, st,
                     (double)ms);
      if (best == 0 || ms < (1.0f - kMargin) * best_ms) {
        best = g;
        best_st = st;
        best_ms = ms;
      }
    }
  } catch (...) {
    toeplitz_set_group(H_, rp_, eb, nslices, 0);
    toeplitz_set_streams(H_, rp_, eb, nslices, 0);
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    throw;
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  toeplitz_set_group(H_, rp_, eb, nslices, best);
  toeplitz_set_streams(H_, rp_, eb, nslices, best_st);
  return best;
}

bool Psf::apply_half(const void* g16, const float* gsc, float* out,
                     int nslices, double* dot_partials, hipStream_t stream,
                     bool wt16) {
  TC_REQUIRE(out != nullptr, "Toeplitz: null output");
  return run_half(g16, gsc, out, nslices, dot_partials, nullptr, stream, wt16);
}

bool Psf::apply_commit_half(const void* g16, const float* gsc,
                            const StepCommit& c, int nslices,
                            double* dot_partials, hipStream_t stream,
                            bool wt16) {
  TC_REQUIRE((c.xp == nullptr) == (c.Tx == nullptr),
             "Toeplitz: xp and Tx must both be given or both be null");
  return run_half(g16, gsc, nullptr, nslices, dot_partials, &c, stream, wt16);
}

bool Psf::apply_commit(const float* g, const StepCommit& c, int nslices,
                       double* dot_partials, hipStream_t stream) {
  TC_REQUIRE(nslices >= 1, "Toeplitz: need at least one slice");
  TC_REQUIRE((c.xp == nullptr) == (c.Tx == nullptr),
             "Toeplitz: xp and Tx must both be given or both be null");
  if (toeplitz_ct_lpw(M_) == 0) return false;
  reserve(nslices);
  const double img_b = 4.0 * nslices * (double)n_ * n_;
  const double spec_b = 8.0 * nslices * (double)n_ * H_;
  return toeplitz_apply_ct(M_, g, nullptr, c.Tdst, work_.as<float2>(),
                           spectrum(), n_, H_, rp_, nslices, 0, dot_partials,
                           stream, img_b, spec_b, &c, streams_for(nslices, 8));
}

void Psf::apply(const float* x, const float* b, float* out, int nslices,
                int mode, double* dot_partials, hipStream_t stream) {
  TC_REQUIRE(nslices >= 1, "Toeplitz: need at least one slice");
  TC_REQUIRE(mode == 0 || (mode == 1 && b != nullptr), "Toeplitz: bad mode");
  reserve(nslices);
  float2* wt = work_.as<float2>();
  // algorithmic bytes: images n^2 floats per slice, spectrum n*H complex
  const double img_b = 4.0 * nslices * (double)n_ * n_;
  const double spec_b = 8.0 * nslices * (double)n_ * H_;
  if (toeplitz_apply_ct(M_, x, b, out, wt, spectrum(), n_, H_, rp_, nslices,
                        mode, dot_partials, stream, img_b, spec_b, nullptr,
                        streams_for(nslices, 8)))
    return;
  apply_generic(x, b, out, nslices, mode, dot_partials, wt, stream);
}

// The runtime-plan passes (FFT lengths without a compile-time plan) on
// workspace wt for nslices slices.
void Psf::apply_generic(const float* x, const float* b, float* out,
                        int nslices, int mode, double* dot_partials,
                        float2* wt, hipStream_t stream) {
  const double img_b = 4.0 * nslices * (double)n_ * n_;
  const double spec_b = 8.0 * nslices * (double)n_ * H_;
  const FFTLength& F = fft_length(M_);
  const int npairs = (n_ + 1) / 2;

  // pass A
  {
    LdsLaunch ll = plan_lds_launch(F, 4, 80 * 1024);
    int nbps = (int)cdiv(npairs, ll.lpw);
    unsigned nblk = (unsigned)nbps * nslices;
    ktimer_begin(KC_TOEPLITZ_ROWS_FWD, stream);
    TC_DISPATCH_NB(ll.nb, {
      auto k = toep_rows_fwd<NB>;
      allow_lds((const void*)k, ll.smem);
      hipLaunchKernelGGL(k, dim3(nblk), dim3(ll.nthr), ll.smem, stream, x, wt,
                         F.plan(), n_, H_, rp_, ll.lpw, nbps);
    });
    TC_HIP(hipGetLastError());
    ktimer_end(KC_TOEPLITZ_ROWS_FWD, stream, img_b + spec_b);
  }
  // pass B
  {
    LdsLaunch ll = plan_lds_launch(F, 1, 80 * 1024);
    int nbps = (int)cdiv(H_, ll.lpw);
    unsigned nblk = (unsigned)nbps * nslices;
    ktimer_begin(KC_TOEPLITZ_COLS, stream);
    TC_DISPATCH_NB(ll.nb, {
      auto k = toep_cols<NB>;
      allow_lds((const void*)k, ll.smem);
      hipLaunchKernelGGL(k, dim3(nblk), dim3(ll.nthr), ll.smem, stream, wt,
                         spectrum(), F.plan(), n_, H_, rp_, ll.lpw, nbps,
                         dot_partials);
    });
    TC_HIP(hipGetLastError());
    ktimer_end(KC_TOEPLITZ_COLS, stream,
               2.0 * spec_b + 4.0 * (double)H_ * M_);
  }
  // pass C
  {
    LdsLaunch ll = plan_lds_launch(F, 4, 80 * 1024);
    int nbps = (int)cdiv(npairs, ll.lpw);
    unsigned nblk = (unsigned)nbps * nslices;
    ktimer_begin(KC_TOEPLITZ_ROWS_INV, stream);
    TC_DISPATCH_NB(ll.nb, {
      if (mode == 0) {
        auto k = toep_rows_inv<NB, 0>;
        allow_lds((const void*)k, ll.smem);
        hipLaunchKernelGGL(k, dim3(nblk), dim3(ll.nthr), ll.smem, stream, wt,
                           b, out, F.plan(), n_, H_, rp_, ll.lpw, nbps);
      } else {
        auto k = toep_rows_inv<NB, 1>;
        allow_lds((const void*)k, ll.smem);
        hipLaunchKernelGGL(k, dim3(nblk), dim3(ll.nthr), ll.smem, stream, wt,
                           b, out, F.plan(), n_, H_, rp_, ll.lpw, nbps);
      }
    });
    TC_HIP(hipGetLastError());
    ktimer_end(KC_TOEPLITZ_ROWS_INV, stream,
               spec_b + img_b * (mode == 1 ? 2.0 : 1.0));
  }
}

void Psf::apply_ws(const float* x, float* out, int nslices,
                   double* dot_partials, void* ws, size_t ws_bytes,
                   hipStream_t stream) {
  TC_REQUIRE(nslices >= 1, "Toeplitz: need at least one slice");
  const size_t per = workspace_bytes_per_slice();
  TC_REQUIRE(ws && ws_bytes >= per, "Toeplitz: workspace of " +
                                        std::to_string(ws_bytes) +
                                        " bytes holds no slice (needs " +
                                        std::to_string(per) + ")");
  const int cap = (int)std::min<size_t>(ws_bytes / per, (size_t)nslices);
  float2* wt = static_cast<float2*>(ws);
  const double img_b = 4.0 * nslices * (double)n_ * n_;
  const double spec_b = 8.0 * nslices * (double)n_ * H_;
  if (toeplitz_apply_ct(M_, x, nullptr, out, wt, spectrum(), n_, H_, rp_,
                        nslices, 0, dot_partials, stream, img_b, spec_b,
                        nullptr, nullptr, cap))
    return;
  // runtime-plan passes, `cap` slices at a time
  const long plane = (long)n_ * n_;
  const int ppart = toeplitz_num_partials(*this, 1);
  for (int s0 = 0; s0 < nslices; s0 += cap) {
    const int ns = std::min(cap, nslices - s0);
    apply_generic(x + s0 * plane, nullptr, out + s0 * plane, ns, 0,
                  dot_partials ? dot_partials + (long)s0 * ppart : nullptr, wt,
                  stream);
  }
}

// number of partial sums written by apply() for `nslices` slices
int toeplitz_num_partials(const Psf& p, int nslices) {
  const int ct = toeplitz_ct_lpw(p.M());
  if (ct > 0) return (int)cdiv(p.H(), ct) * nslices;
  const FFTLength& F = fft_length(p.M());
  LdsLaunch ll = plan_lds_launch(F, 1, 80 * 1024);
  return (int)cdiv(p.H(), ll.lpw) * nslices;
}

}  // namespace tc
