// Line transforms of any 2,3,5,7-smooth length on radices chosen at run time.
#pragma once

#include "fft_ct.h"

namespace tc {

// Any 2,3,5,7-smooth length as two to six radices of up to 16,
// lines in LDS, each stage from one buffer to the other (one barrier a stage).
// The former form took radices 8, 4, 2, 3, 5, 7 in place: four to six stages
// of two barriers each (3 x 672 lines of 672 points: 25 -> 17 us for the 337
// columns of the half grid, 12 us for the packed rows).
// Lines too long for two buffers (more than about 9900 points) run in place.
// ---------------------------------------------------------------------------

constexpr int RT_MAX_THREADS = 512;
constexpr int RT_MAX_STAGES = 8;

struct RtPlan {
  int L, nst, ldl;  // ldl: LDS elements per line and buffer
  int lines_off;    // elements from one buffer to the other
  int radix[RT_MAX_STAGES];
  const float2* tw;  // exp(-2 pi i m / L)
};

// one unused slot per 32: the first stages' strided stores spread over banks
__host__ __device__ __forceinline__ int rt_pad(int i) { return i + (i >> 5); }

template <int R, int DIR>
__device__ __forceinline__ void rt_stage(const float2* in, float2* out,
                                         int nlines, const RtPlan& P, int Ns,
                                         int tid, int nthr) {
  const int nb = P.L / R, step = P.L / (Ns * R);
  for (int t = tid; t < nlines * nb; t += nthr) {
    const int line = nlines == 1 ? 0 : t / nb;
    const int j = t - line * nb;
    const int k = Ns == 1 ? 0 : j % Ns;
    const float2* src = in + line * P.ldl;
    float2 v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = src[rt_pad(j + r * nb)];
    if (Ns > 1) {
#pragma unroll
      for (int r = 1; r < R; ++r) {
        const float2 w = P.tw[k * r * step];
        v[r] = DIR < 0 ? cmul(v[r], w) : cmulc(v[r], w);
      }
    }
    ct::DftC<R, DIR>::run(v);
    float2* dst = out + line * P.ldl;
    const int d = (j - k) * R + k;
#pragma unroll
    for (int r = 0; r < R; ++r) dst[rt_pad(d + r * Ns)] = v[r];
  }
}

// Transforms the lines in the first buffer of `sm` (the second if `second`)
// and returns the buffer that holds the result.  Called by every thread, with
// the data behind a barrier; returns behind one.
template <int DIR>
__device__ __forceinline__ float2* rt_fft(float2* sm, int nlines,
                                          const RtPlan& P, int tid, int nthr,
                                          bool second = false) {
  float2* a = second ? sm + P.lines_off : sm;
  float2* b = second ? sm : sm + P.lines_off;
  int Ns = 1;
  for (int s = 0; s < P.nst; ++s) {
    const int R = P.radix[s];
    switch (R) {
#define TC_RT(RR)                                         \
  case RR:                                                \
    rt_stage<RR, DIR>(a, b, nlines, P, Ns, tid, nthr);    \
    break;
      TC_RT(2) TC_RT(3) TC_RT(4) TC_RT(5) TC_RT(6) TC_RT(7) TC_RT(8) TC_RT(9)
      TC_RT(10) TC_RT(12) TC_RT(14) TC_RT(15) TC_RT(16)
#undef TC_RT
    }
    __syncthreads();
    Ns *= R;
    float2* t = a;
    a = b;
    b = t;
  }
  return a;
}

struct RtLaunch {
  RtPlan plan;
  int lpw, nthr;
  size_t smem;
};

// Whether a line fits LDS in two buffers, and the launch shape for lines of
// length L: at most `want` lines per workgroup, 64 KB of LDS or one line, and a
// thread per butterfly of the smallest radix up to RT_MAX_THREADS.
bool rt_fits(int L);
RtLaunch rt_launch(int L, long nlines, int want);

}  // namespace tc
