// Batched line transforms on compile-time plans (fft_ct.h) for the lengths the
// NUFFT fine grids, the ray transforms and the PSF spectra use.  One workgroup
// transforms LPW whole lines: every element is loaded into registers, the
// stages exchange through one padded LDS line per line, and the outputs are
// stored from registers, so a line is read and written once.  The kernels are
// templates; each fft_lines_ct_<k>.hip instantiates some of the lengths, and
// lengths without a plan fall back to the runtime-plan kernels.
#pragma once

#include <algorithm>

#include "fft_ct.h"
#include "fft_ops.h"
#include "lds_launch.h"

namespace tc {

namespace {

using ct::Radices;

// Line stride (elements) for `lines` lines of `elems` padded elements:
// congruent to ceil(32 / lines) modulo 32, so that the lines of a
// workgroup start on different LDS banks.
constexpr int lines_stride(int elems, int lines) {
  if (lines <= 1) return elems;
  const int target = (32 + lines - 1) / lines % 32;
  return elems + (((target - elems) % 32) + 32) % 32;
}

template <class Rad>
struct RadixOps;
template <int... Rs>
struct RadixOps<Radices<Rs...>> {
  static constexpr int first = ct::RadixList<Rs...>::at(0);
  static constexpr int last = ct::RadixList<Rs...>::at(sizeof...(Rs) - 1);
  template <int L>
  static constexpr int elems() { return ct::line_elems<L, Rs...>(); }
  template <int L, int E, int DIR>
  __device__ __forceinline__ static void run(float2* v, float2* line, int t,
                                             bool active,
                                             const float2* __restrict__ tw) {
    ct::transform<L, E, DIR, false, Rs...>(v, line, t, active, tw);
  }
};

// Fwd: the radices of the line transforms (either direction); Inv: the
// same radices reversed, for a forward-multiply-inverse sequence held in
// registers (the inverse's first-stage inputs are the forward's outputs).
template <int L_, int E_, int LPW_, class Fwd, class Inv>
struct LinePlan {
  static constexpr int L = L_, E = E_, LPW = LPW_, T = L_ / E_;
  static constexpr int NT = LPW_ * T;
  static constexpr int LE = RadixOps<Fwd>::template elems<L_>() >
                                    RadixOps<Inv>::template elems<L_>()
                                ? RadixOps<Fwd>::template elems<L_>()
                                : RadixOps<Inv>::template elems<L_>();
  static constexpr int LS = lines_stride(LE, LPW_);
  static constexpr int R1 = RadixOps<Fwd>::first;
  static constexpr int RS = RadixOps<Fwd>::last;
  static_assert(RadixOps<Inv>::first == RS && RadixOps<Inv>::last == R1,
                "Inv must be Fwd reversed");
  static const float2* twiddles() { return ct::plan_twiddles<Fwd, Inv>(); }
  template <int DIR>
  __device__ __forceinline__ static void run(float2* v, float2* line, int t,
                                             bool active,
                                             const float2* __restrict__ tw) {
    RadixOps<Fwd>::template run<L_, E_, DIR>(v, line, t, active, tw);
  }
  __device__ __forceinline__ static void run_inv(float2* v, float2* line,
                                                 int t, bool active,
                                                 const float2* __restrict__ tw) {
    RadixOps<Inv>::template run<L_, E_, 1>(v, line, t, active,
                                           tw + ct::tw_count<Fwd>);
  }
};

// Line l of batch b starts at b * bstride + (l / lgroup) * lstride + l %
// lgroup; element i at + i * estride.  Of a line, the elements [0, nin) and [L
// - nin_hi, L) are read (the others are zero) and [0, nout) and [L - nout_hi,
// L) written.  COL: the workgroup's lines are adjacent columns, so consecutive
// threads take consecutive lines (coalesced loads of a row); otherwise
// consecutive threads take consecutive elements of one line.
template <class P, int DIR, bool COL>
__global__ void __launch_bounds__(P::NT)
ct_lines_kernel(const float2* in, float2* out, const float2* __restrict__ tw,
                int lines_per_batch, long nlines, long bstride, long lstride,
                int lgroup, long estride, int nin, int nin_hi, int nout, int nout_hi,
                float scale) {
  extern __shared__ float2 sm[];
  constexpr int L = P::L, E = P::E, T = P::T, LPW = P::LPW;
  constexpr int R1 = P::R1, RS = P::RS;
  const int line = COL ? (int)(threadIdx.x % LPW) : (int)(threadIdx.x / T);
  const int t = COL ? (int)(threadIdx.x / LPW) : (int)(threadIdx.x % T);
  const long gl = (long)xcd_remap(blockIdx.x, gridDim.x) * LPW + line;
  const bool active = gl < nlines;
  const long b = active ? gl / lines_per_batch : 0;
  const int lb = active ? (int)(gl - b * lines_per_batch) : 0;
  const long base = b * bstride + (lb / lgroup) * lstride + lb % lgroup;
  float2 v[E];
#pragma unroll
  for (int i = 0; i < E / R1; ++i)
#pragma unroll
    for (int r = 0; r < R1; ++r) {
      const int idx = t + i * T + r * (L / R1);
      v[i * R1 + r] = (active && (idx < nin || idx >= L - nin_hi))
                          ? in[base + idx * estride]
                          : make_float2(0.f, 0.f);
    }
  // every load of the workgroup precedes the transform's first barrier,
  // and the workgroup's lines are its own: in == out is safe
  P::template run<DIR>(v, sm + line * P::LS, t, active, tw);
  if (!active) return;
#pragma unroll
  for (int i = 0; i < E / RS; ++i)
#pragma unroll
    for (int r = 0; r < RS; ++r) {
      const int idx = t + i * T + r * (L / RS);
      if (idx < nout || idx >= L - nout_hi) {
        const float2 q = v[i * RS + r];
        out[base + idx * estride] = make_float2(q.x * scale, q.y * scale);
      }
    }
}

template <class P, int DIR, bool COL>
void launch_ct_lines(const LineFFTArgs& a, hipStream_t stream) {
  const long nlines = (long)a.lines_per_batch * a.nbatch;
  if (nlines == 0) return;
  const size_t smem = sizeof(float2) * (size_t)P::LPW * P::LS;
  auto k = ct_lines_kernel<P, DIR, COL>;
  allow_lds((const void*)k, smem);
  const unsigned nblk = (unsigned)cdiv(nlines, P::LPW);
  hipLaunchKernelGGL(k, dim3(nblk), dim3(P::NT), smem, stream, a.in, a.out,
                     P::twiddles(), a.lines_per_batch, nlines,
                     a.bstride, a.lstride, a.lgroup, a.estride, a.nin, a.nin_hi, a.nout,
                     a.nout_hi, a.scale);
  TC_HIP(hipGetLastError());
}

template <class P>
void run_lines(const LineFFTArgs& a, int dir, hipStream_t stream) {
  if (a.colmajor) {
    if (dir < 0) launch_ct_lines<P, -1, true>(a, stream);
    else launch_ct_lines<P, 1, true>(a, stream);
  } else {
    if (dir < 0) launch_ct_lines<P, -1, false>(a, stream);
    else launch_ct_lines<P, 1, false>(a, stream);
  }
}

// ---------------------------------------------------------------------------
// real rows <-> half spectrum (RealRowsArgs, fft_ops.h).  Two rows of one
// slice make one complex line, so a row costs half a complex transform and
// the half spectrum half the memory; the corrections of the NUFFT modes are
// applied on the way.  8 x 1024^2 on a 2048^2 grid: correction and padding
// (95 us) and complex row transforms (90 us) -> 35 us.
// ---------------------------------------------------------------------------

template <class P>
__global__ void __launch_bounds__(P::NT)
ct_r2c_rows_kernel(RealRowsArgs a, const float2* __restrict__ tw) {
  extern __shared__ float2 sm[];
  constexpr int L = P::L, E = P::E, T = P::T, LPW = P::LPW;
  constexpr int R1 = P::R1, RS = P::RS, H = L / 2 + 1;
  const int line = (int)(threadIdx.x / T), t = (int)(threadIdx.x % T);
  const int npair = (a.nm + 1) / 2;
  const long g0 = (long)xcd_remap(blockIdx.x, gridDim.x) * LPW;
  const long nlines = (long)a.nsl * npair;
  const int lo = (a.nm + 1) / 2, hi = a.nm / 2;
  {
    const long gl = g0 + line;
    const bool active = gl < nlines;
    const long s = active ? gl / npair : 0;
    const int ka = active ? 2 * (int)(gl - s * npair) : 0;
    const bool hasb = ka + 1 < a.nm;
    const float ca = a.corr[ka], cb = hasb ? a.corr[ka + 1] : 0.f;
    const float* f = a.real_in + (s * a.nm + ka) * a.nm;
    float2 v[E];
#pragma unroll
    for (int i = 0; i < E / R1; ++i)
#pragma unroll
      for (int r = 0; r < R1; ++r) {
        const int idx = t + i * T + r * (L / R1);
        float2 w = make_float2(0.f, 0.f);
        if (active && (idx < lo || idx >= L - hi)) {
          const int k = idx < lo ? idx + hi : idx - (L - hi);
          const float c = a.corr[k];
          w.x = f[k] * c * ca;
          if (hasb) w.y = f[a.nm + k] * c * cb;
        }
        v[i * R1 + r] = w;
      }
    float2* ln = sm + line * P::LS;
    P::template run<-1>(v, ln, t, true, tw);
#pragma unroll
    for (int i = 0; i < E / RS; ++i)
#pragma unroll
      for (int r = 0; r < RS; ++r) ln[t + i * T + r * (L / RS)] = v[i * RS + r];
  }
  __syncthreads();
  // two columns of both rows a thread: 16-byte stores, consecutive threads
  // along a block's columns, then along the workgroup's row pairs
  constexpr int HC = HG_B / 2, NC = (H + HG_B - 1) / HG_B * HC;
  for (int q = threadIdx.x; q < LPW * NC; q += P::NT) {
    const int l = q / HC % LPW;
    const int k = (q / (HC * LPW) * HC + q % HC) * 2;
    const long gl = g0 + l;
    if (k >= H || gl >= nlines) continue;
    const long s = gl / npair;
    const int ka = 2 * (int)(gl - s * npair);
    const int ra = ka < hi ? L + ka - hi : ka - hi;
    const int rb = ka + 1 < hi ? L + ka + 1 - hi : ka + 1 - hi;
    float4 fa, fb;  // column H, if any, is in the block's padding
    {
      const float2 zk = sm[l * P::LS + k];
      const float2 zm = cconj(sm[l * P::LS + (k == 0 ? 0 : L - k)]);
      const float2 sp = cadd(zk, zm), df = csub(zk, zm);
      fa.x = 0.5f * sp.x, fa.y = 0.5f * sp.y;
      fb.x = 0.5f * df.y, fb.y = -0.5f * df.x;
    }
    {
      const float2 zk = sm[l * P::LS + k + 1];
      const float2 zm = cconj(sm[l * P::LS + L - k - 1]);
      const float2 sp = cadd(zk, zm), df = csub(zk, zm);
      fa.z = 0.5f * sp.x, fa.w = 0.5f * sp.y;
      fb.z = 0.5f * df.y, fb.w = -0.5f * df.x;
    }
    float2* half = a.half + s * half_grid_size(L);
    *reinterpret_cast<float4*>(half + half_at(L, ra, k)) = fa;
    if (ka + 1 < a.nm) *reinterpret_cast<float4*>(half + half_at(L, rb, k)) = fb;
  }
}

template <class P>
__global__ void __launch_bounds__(P::NT)
ct_c2r_rows_kernel(RealRowsArgs a, const float2* __restrict__ tw) {
  extern __shared__ float2 sm[];
  constexpr int L = P::L, E = P::E, T = P::T, LPW = P::LPW;
  constexpr int R1 = P::R1, RS = P::RS, H = L / 2 + 1;
  const int npair = (a.nm + 1) / 2;
  const long g0 = (long)xcd_remap(blockIdx.x, gridDim.x) * LPW;
  const long nlines = (long)a.nsl * npair;
  const int lo = (a.nm + 1) / 2, hi = a.nm / 2;
  // two columns of both rows a thread, consecutive threads along a block's
  // columns, then along the workgroup's row pairs; every load of the thread in
  // flight at once, then the LDS writes
  constexpr int HC = HG_B / 2, NC = (H + HG_B - 1) / HG_B * HC;
  constexpr int NQ = (LPW * NC + P::NT - 1) / P::NT;
  float4 wa[NQ], wb[NQ];
#pragma unroll
  for (int j = 0; j < NQ; ++j) {
    const int q = (int)threadIdx.x + j * P::NT;
    const int l = q / HC % LPW;
    const int k = (q / (HC * LPW) * HC + q % HC) * 2;
    const long gl = g0 + l;
    wa[j] = wb[j] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (k < H && gl < nlines) {
      const long s = gl / npair;
      const int ka = 2 * (int)(gl - s * npair);
      const int ra = ka < hi ? L + ka - hi : ka - hi;
      const int rb = ka + 1 < hi ? L + ka + 1 - hi : ka + 1 - hi;
      const float2* half = a.half + s * half_grid_size(L);
      wa[j] = *reinterpret_cast<const float4*>(half + half_at(L, ra, k));
      if (ka + 1 < a.nm)
        wb[j] = *reinterpret_cast<const float4*>(half + half_at(L, rb, k));
    }
  }
#pragma unroll
  for (int j = 0; j < NQ; ++j) {
    const int q = (int)threadIdx.x + j * P::NT;
    const int l = q / HC % LPW;
    const int k0 = (q / (HC * LPW) * HC + q % HC) * 2;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int k = k0 + e;
      if (k >= H) break;
      float2 x = e ? make_float2(wa[j].z, wa[j].w)
                   : make_float2(wa[j].x, wa[j].y);
      float2 y = e ? make_float2(wb[j].z, wb[j].w)
                   : make_float2(wb[j].x, wb[j].y);
      if (k == 0 || 2 * k == L) x.y = y.y = 0.f;  // real by symmetry
      sm[l * P::LS + k] = make_float2(x.x - y.y, x.y + y.x);
      if (k > 0 && L - k >= H)
        sm[l * P::LS + L - k] = make_float2(x.x + y.y, y.x - x.y);
    }
  }
  __syncthreads();
  const int line = (int)(threadIdx.x / T), t = (int)(threadIdx.x % T);
  float2* ln = sm + line * P::LS;
  float2 v[E];
#pragma unroll
  for (int i = 0; i < E / R1; ++i)
#pragma unroll
    for (int r = 0; r < R1; ++r) v[i * R1 + r] = ln[t + i * T + r * (L / R1)];
  __syncthreads();
  P::template run<1>(v, ln, t, true, tw);
  const long gl = g0 + line;
  if (gl >= nlines) return;
  const long s = gl / npair;
  const int ka = 2 * (int)(gl - s * npair);
  const bool hasb = ka + 1 < a.nm;
  const float ca = a.corr[ka] * a.scale;
  const float cb = hasb ? a.corr[ka + 1] * a.scale : 0.f;
  float* o = a.real_out + (s * a.nm + ka) * a.nm;
#pragma unroll
  for (int i = 0; i < E / RS; ++i)
#pragma unroll
    for (int r = 0; r < RS; ++r) {
      const int idx = t + i * T + r * (L / RS);
      if (idx < lo || idx >= L - hi) {
        const int k = idx < lo ? idx + hi : idx - (L - hi);
        const float c = a.corr[k];
        o[k] = v[i * RS + r].x * c * ca;
        if (hasb) o[a.nm + k] = v[i * RS + r].y * c * cb;
      }
    }
}

template <class P>
void run_real_rows(const RealRowsArgs& a, bool r2c, hipStream_t stream) {
  const long nlines = (long)a.nsl * ((a.nm + 1) / 2);
  if (nlines == 0) return;
  const size_t smem = sizeof(float2) * (size_t)P::LPW * P::LS;
  const unsigned nblk = (unsigned)cdiv(nlines, P::LPW);
  const float2* tw = P::twiddles();
  auto k = r2c ? ct_r2c_rows_kernel<P> : ct_c2r_rows_kernel<P>;
  allow_lds((const void*)k, smem);
  hipLaunchKernelGGL(k, dim3(nblk), dim3(P::NT), smem, stream, a, tw);
  TC_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------
// Centred chirp-z (Bluestein) DFT of rays of N samples on a planned length
// L >= 2N - 1 (RayArgs, fft_ops.h).  Two rays of one slice make one complex
// line; the forward transform, the multiply by the chirp's spectrum and the
// inverse (radices reversed, so its inputs are the forward's outputs) stay in
// registers.
// ---------------------------------------------------------------------------

template <class P, bool TO_HALF>
__global__ void __launch_bounds__(P::NT)
ct_ray_kernel(RayArgs a, const float2* __restrict__ tw) {
  extern __shared__ float2 sm[];
  constexpr int L = P::L, E = P::E, T = P::T, LPW = P::LPW;
  constexpr int R1 = P::R1, RS = P::RS;
  const int line = (int)(threadIdx.x / T);
  const int t = (int)(threadIdx.x % T);
  const int npair = (a.P + 1) / 2;
  const long g0 = (long)xcd_remap(blockIdx.x, gridDim.x) * LPW;
  const long nlines = (long)a.nsl * npair;
  const long gl = g0 + line;
  const bool active = gl < nlines;
  const long s = active ? gl / npair : 0;
  const int pa = active ? 2 * (int)(gl - s * npair) : 0;
  const bool hasb = active && pa + 1 < a.P;
  const int N = a.N, c = N / 2;
  float2 level = make_float2(0.f, 0.f);
  if constexpr (TO_HALF) {
    const float* p = a.real_in + (s * a.P + pa) * N;
    if (active) level.x = ray_level(a, p);
    if (hasb) level.y = ray_level(a, p + N);
  }
  float2 v[E];
#pragma unroll
  for (int i = 0; i < E / R1; ++i)
#pragma unroll
    for (int r = 0; r < R1; ++r) {
      const int idx = t + i * T + r * (L / R1);
      float2 w = make_float2(0.f, 0.f);
      if (active && idx < N) {
        if constexpr (TO_HALF) {
          const float* p = a.real_in + (s * a.P + pa) * N + idx;
          w.x = p[0] - level.x;
          if (hasb) w.y = p[N] - level.y;
        } else {
          const float2* p = a.half_in + (s * a.P + pa) * a.nh;
          w = ray_pair_sample(p, hasb ? p + a.nh : nullptr, idx - c, N);
        }
        w = cmul(w, a.chirp[idx]);
      }
      v[i * R1 + r] = w;
    }
  float2* ln = sm + line * P::LS;
  P::template run<-1>(v, ln, t, true, tw);
#pragma unroll
  for (int i = 0; i < E / RS; ++i)
#pragma unroll
    for (int r = 0; r < RS; ++r) {
      const int k = t + i * T + r * (L / RS);
      v[i * RS + r] = cmul(v[i * RS + r], a.bhat[k]);
    }
  P::run_inv(v, ln, t, true, tw);
  if constexpr (!TO_HALF) {
    if (!active) return;
    float* o = a.real_out + (s * a.P + pa) * N;
#pragma unroll
    for (int i = 0; i < E / R1; ++i)
#pragma unroll
      for (int r = 0; r < R1; ++r) {
        const int j = t + i * T + r * (L / R1);
        if (j < N) {
          const float2 q = cmul(v[i * R1 + r], a.chirp[j]);
          o[j] = q.x * a.scale;
          if (hasb) o[N + j] = q.y * a.scale;
        }
      }
  } else {
#pragma unroll
    for (int i = 0; i < E / R1; ++i)
#pragma unroll
      for (int r = 0; r < R1; ++r) {
        const int j = t + i * T + r * (L / R1);
        if (j < N) ln[j] = cmul(v[i * R1 + r], a.chirp[j]);
      }
    __syncthreads();
    for (int q = threadIdx.x; q < LPW * a.nh; q += P::NT) {
      const int l = q / a.nh, m = q - l * a.nh;
      if (g0 + l >= nlines) break;
      const float2* z = sm + l * P::LS;
      ray_store_pair(a, g0 + l, z[c + m < N ? c + m : 0], z[c - m], m);
    }
  }
}

// Rays of a planned length N == L: one transform instead of two of twice the
// length.  Index i of the line is sample i, or i - N past the middle.
template <class P, bool TO_HALF>
__global__ void __launch_bounds__(P::NT)
ct_ray_direct_kernel(RayArgs a, const float2* __restrict__ tw) {
  extern __shared__ float2 sm[];
  constexpr int N = P::L, E = P::E, T = P::T, LPW = P::LPW, c = N / 2;
  constexpr int R1 = P::R1, RS = P::RS;
  const int line = (int)(threadIdx.x / T);
  const int t = (int)(threadIdx.x % T);
  const int npair = (a.P + 1) / 2;
  const long g0 = (long)xcd_remap(blockIdx.x, gridDim.x) * LPW;
  const long nlines = (long)a.nsl * npair;
  const long gl = g0 + line;
  const bool active = gl < nlines;
  const long s = active ? gl / npair : 0;
  const int pa = active ? 2 * (int)(gl - s * npair) : 0;
  const bool hasb = active && pa + 1 < a.P;
  float2 level = make_float2(0.f, 0.f);
  if constexpr (TO_HALF) {
    const float* p = a.real_in + (s * a.P + pa) * N;
    if (active) level.x = ray_level(a, p);
    if (hasb) level.y = ray_level(a, p + N);
  }
  float2 v[E];
#pragma unroll
  for (int i = 0; i < E / R1; ++i)
#pragma unroll
    for (int r = 0; r < R1; ++r) {
      const int idx = t + i * T + r * (N / R1);
      float2 w = make_float2(0.f, 0.f);
      if (active) {
        if constexpr (TO_HALF) {
          const float* p =
              a.real_in + (s * a.P + pa) * N + (idx < N - c ? idx + c
                                                            : idx - (N - c));
          w.x = p[0] - level.x;
          if (hasb) w.y = p[N] - level.y;
        } else {
          const float2* p = a.half_in + (s * a.P + pa) * a.nh;
          w = ray_pair_sample(p, hasb ? p + a.nh : nullptr,
                              idx < N - c ? idx : idx - N, N);
        }
      }
      v[i * R1 + r] = w;
    }
  float2* ln = sm + line * P::LS;
  P::template run<TO_HALF ? -1 : 1>(v, ln, t, true, tw);
  if constexpr (!TO_HALF) {
    if (!active) return;
    float* o = a.real_out + (s * a.P + pa) * N;
#pragma unroll
    for (int i = 0; i < E / RS; ++i)
#pragma unroll
      for (int r = 0; r < RS; ++r) {
        const int idx = t + i * T + r * (N / RS);
        const int j = idx < N - c ? idx + c : idx - (N - c);
        o[j] = v[i * RS + r].x * a.scale;
        if (hasb) o[N + j] = v[i * RS + r].y * a.scale;
      }
  } else {
#pragma unroll
    for (int i = 0; i < E / RS; ++i)
#pragma unroll
      for (int r = 0; r < RS; ++r) {
        const int idx = t + i * T + r * (N / RS);
        ln[idx < N - c ? idx + c : idx - (N - c)] = v[i * RS + r];
      }
    __syncthreads();
    for (int q = threadIdx.x; q < LPW * a.nh; q += P::NT) {
      const int l = q / a.nh, m = q - l * a.nh;
      if (g0 + l >= nlines) break;
      const float2* z = sm + l * P::LS;
      ray_store_pair(a, g0 + l, z[c + m < N ? c + m : 0], z[c - m], m);
    }
  }
}

template <class P>
void run_rays(const RayArgs& a, bool to_half, hipStream_t stream) {
  const long nlines = (long)a.nsl * ((a.P + 1) / 2);
  if (nlines == 0) return;
  const size_t smem = sizeof(float2) * (size_t)P::LPW * P::LS;
  const unsigned nblk = (unsigned)cdiv(nlines, P::LPW);
  const float2* tw = P::twiddles();
  auto k = a.N == a.L ? (to_half ? ct_ray_direct_kernel<P, true>
                                 : ct_ray_direct_kernel<P, false>)
                      : (to_half ? ct_ray_kernel<P, true>
                                 : ct_ray_kernel<P, false>);
  allow_lds((const void*)k, smem);
  hipLaunchKernelGGL(k, dim3(nblk), dim3(P::NT), smem, stream, a, tw);
  TC_HIP(hipGetLastError());
}

}  // namespace

// The transforms of one planned length.
struct LineOps {
  int L;
  void (*lines)(const LineFFTArgs&, int dir, hipStream_t);
  void (*real_rows)(const RealRowsArgs&, bool r2c, hipStream_t);
  void (*rays)(const RayArgs&, bool to_half, hipStream_t);
  const float2* (*twiddles)();
};

// Plans, ascending: length, elements per thread, lines per workgroup and
// radices (each divides the elements per thread).  From 192 on the lengths are
// at most 1/8 apart, but for 216 to 256, 324 to 384 and 648 to 768 (18.5 %), so
// that a chirp length rounded up to one costs little; radices of 8 to 36 keep
// the LDS exchanges at one to three.
#define TC_FOR_LINE_LENGTHS_1(X) \
  X(64) X(96) X(128) X(144) X(192) X(216) X(256) X(288) X(324) X(384) X(432)
#define TC_FOR_LINE_LENGTHS_2(X) \
  X(486) X(512) X(576) X(648) X(768) X(864) X(972) X(1024) X(1152) X(1296)
#define TC_FOR_LINE_LENGTHS_3(X) \
  X(1458) X(1536) X(1728) X(1944) X(2048) X(2304) X(2592) X(2916) X(3072)
#define TC_FOR_LINE_LENGTHS_4(X) \
  X(3456) X(3888) X(4096) X(4374) X(4608) X(5184) X(5832) X(6144)
#define TC_FOR_LINE_LENGTHS_5(X) \
  X(6912) X(7776) X(8192) X(8748) X(9216) X(10368) X(11664)
#define TC_FOR_LINE_LENGTHS(X)                          \
  TC_FOR_LINE_LENGTHS_1(X) TC_FOR_LINE_LENGTHS_2(X)     \
  TC_FOR_LINE_LENGTHS_3(X) TC_FOR_LINE_LENGTHS_4(X)     \
  TC_FOR_LINE_LENGTHS_5(X)
#define TC_LINE_OPS_DECL(LL) extern LineOps kLineOps##LL;
TC_FOR_LINE_LENGTHS(TC_LINE_OPS_DECL)
#undef TC_LINE_OPS_DECL

namespace {
using L64 = LinePlan<64, 8, 32, Radices<8, 8>, Radices<8, 8>>;
using L96 = LinePlan<96, 24, 32, Radices<12, 8>, Radices<8, 12>>;
using L128 = LinePlan<128, 16, 32, Radices<16, 8>, Radices<8, 16>>;
using L144 = LinePlan<144, 12, 16, Radices<12, 12>, Radices<12, 12>>;
using L192 = LinePlan<192, 24, 32, Radices<24, 8>, Radices<8, 24>>;
using L216 = LinePlan<216, 12, 12, Radices<12, 6, 3>, Radices<3, 6, 12>>;
using L256 = LinePlan<256, 16, 16, Radices<16, 16>, Radices<16, 16>>;
using L288 = LinePlan<288, 24, 16, Radices<24, 12>, Radices<12, 24>>;
using L324 = LinePlan<324, 18, 12, Radices<18, 18>, Radices<18, 18>>;
using L384 = LinePlan<384, 24, 16, Radices<24, 8, 2>, Radices<2, 8, 24>>;
using L432 = LinePlan<432, 12, 6, Radices<12, 12, 3>, Radices<3, 12, 12>>;
using L486 = LinePlan<486, 18, 9, Radices<18, 9, 3>, Radices<3, 9, 18>>;
using L512 = LinePlan<512, 8, 4, Radices<8, 8, 8>, Radices<8, 8, 8>>;
using L576 = LinePlan<576, 24, 10, Radices<24, 24>, Radices<24, 24>>;
using L648 = LinePlan<648, 18, 6, Radices<18, 18, 2>, Radices<2, 18, 18>>;
using L768 = LinePlan<768, 24, 8, Radices<24, 8, 4>, Radices<4, 8, 24>>;
using L864 = LinePlan<864, 24, 6, Radices<24, 12, 3>, Radices<3, 12, 24>>;
using L972 = LinePlan<972, 18, 4, Radices<18, 18, 3>, Radices<3, 18, 18>>;
using L1024 = LinePlan<1024, 16, 4, Radices<16, 16, 4>, Radices<4, 16, 16>>;
using L1152 = LinePlan<1152, 24, 4, Radices<24, 24, 2>, Radices<2, 24, 24>>;
using L1296 = LinePlan<1296, 36, 6, Radices<36, 36>, Radices<36, 36>>;
using L1458 = LinePlan<1458, 18, 3, Radices<18, 9, 9>, Radices<9, 9, 18>>;
using L1536 = LinePlan<1536, 24, 4, Radices<24, 8, 8>, Radices<8, 8, 24>>;
using L1728 = LinePlan<1728, 24, 3, Radices<24, 24, 3>, Radices<3, 24, 24>>;
using L1944 = LinePlan<1944, 18, 2, Radices<18, 18, 6>, Radices<6, 18, 18>>;
using L2048 = LinePlan<2048, 16, 2, Radices<16, 16, 8>, Radices<8, 16, 16>>;
using L2304 = LinePlan<2304, 24, 2, Radices<24, 24, 4>, Radices<4, 24, 24>>;
using L2592 = LinePlan<2592, 36, 3, Radices<18, 12, 12>, Radices<12, 12, 18>>;
using L2916 = LinePlan<2916, 18, 2, Radices<18, 18, 9>, Radices<9, 18, 18>>;
using L3072 = LinePlan<3072, 24, 2, Radices<24, 8, 4, 4>, Radices<4, 4, 8, 24>>;
using L3456 = LinePlan<3456, 24, 2, Radices<24, 24, 6>, Radices<6, 24, 24>>;
using L3888 = LinePlan<3888, 36, 2, Radices<18, 18, 12>, Radices<12, 18, 18>>;
using L4096 = LinePlan<4096, 16, 1, Radices<16, 16, 16>, Radices<16, 16, 16>>;
using L4374 = LinePlan<4374, 18, 2, Radices<18, 9, 9, 3>, Radices<3, 9, 9, 18>>;
using L4608 = LinePlan<4608, 24, 1, Radices<24, 24, 8>, Radices<8, 24, 24>>;
using L5184 = LinePlan<5184, 36, 1, Radices<36, 12, 12>, Radices<12, 12, 36>>;
using L5832 = LinePlan<5832, 18, 1, Radices<18, 18, 18>, Radices<18, 18, 18>>;
using L6144 = LinePlan<6144, 24, 1, Radices<24, 8, 8, 4>, Radices<4, 8, 8, 24>>;
using L6912 = LinePlan<6912, 24, 1, Radices<24, 24, 12>, Radices<12, 24, 24>>;
using L7776 = LinePlan<7776, 36, 1, Radices<36, 18, 12>, Radices<12, 18, 36>>;
using L8192 = LinePlan<8192, 32, 1, Radices<32, 16, 16>, Radices<16, 16, 32>>;
using L8748 =
    LinePlan<8748, 18, 1, Radices<18, 18, 9, 3>, Radices<3, 9, 18, 18>>;
using L9216 =
    LinePlan<9216, 24, 1, Radices<24, 24, 4, 4>, Radices<4, 4, 24, 24>>;
using L10368 =
    LinePlan<10368, 36, 1, Radices<36, 12, 12, 2>, Radices<2, 12, 12, 36>>;
using L11664 = LinePlan<11664, 36, 1, Radices<36, 18, 18>, Radices<18, 18, 36>>;
}  // namespace

#define TC_LINE_OPS_DEF(LL)                                             \
  LineOps kLineOps##LL = {LL, run_lines<L##LL>, run_real_rows<L##LL>, \
                                run_rays<L##LL>, L##LL::twiddles};

}  // namespace tc
