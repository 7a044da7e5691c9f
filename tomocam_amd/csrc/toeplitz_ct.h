// Toeplitz passes on compile-time FFT plans (fft_ct.h): the kernels and their
// launches.  toeplitz_ct.hip instantiates the plans that have the
// mixed-precision forms, toeplitz_plain_<k>.hip the FP32-only ones; lengths
// without a plan use the runtime-plan kernels in toeplitz.hip.
#pragma once

#include <hip/hip_fp16.h>

#include <algorithm>

#include "fft_ct.h"
#include "lds_launch.h"
#include "toeplitz.h"

namespace tc {

// Slices per group of passes (toeplitz_ct.hip).
int toeplitz_group_slices(int nslices, int H, int rp, int elem_bytes);

using ct::Radices;

template <int L, int E, int DIR, class Rad>
struct Xform;
template <int L, int E, int DIR, int... Rs>
struct Xform<L, E, DIR, Radices<Rs...>> {
  static constexpr int first = ct::RadixList<Rs...>::at(0);
  static constexpr int last = ct::RadixList<Rs...>::at(sizeof...(Rs) - 1);
  // ZIN: input zero from index L/2 on (every line here is zero-padded
  // from n <= L/2), so the first stage skips those terms
  template <bool ZIN = false>
  __device__ __forceinline__ static void run(float2* v, float2* line, int t,
                                             bool active,
                                             const float2* __restrict__ tw) {
    // the zero-upper DFT form needs a radix-2 first factor; other first
    // radices still skip the padding's loads and compute on zeros
    constexpr bool z = ZIN && ct::first_radix<first>() == 2;
    ct::transform<L, E, DIR, z, Rs...>(v, line, t, active, tw);
  }
};

// Zero padding: a line holds n <= L/2 data values (L >= 2n - 1, L even).
// Element r of a radix-R butterfly sits at index j + r L/R with
// j < L/R, so for r >= R/2 it lies in the padding: stage-1 inputs there are
// zero and last-stage outputs there are not kept.

// Plans: forward radices Fwd, inverse radices Inv = reversed Fwd, LPW lines
// per workgroup in the row passes and LPWC in the column pass.  ZA: pass A
// skips the zero padding of its input in the first FFT stage.
template <int L, class Rad>
struct LineElems;
template <int L, int... Rs>
struct LineElems<L, Radices<Rs...>> {
  static constexpr int value = ct::line_elems<L, Rs...>();
};

// Stride between the LDS lines of a workgroup with `lines` lines: at least
// `elems`, and congruent to ceil(32 / lines) modulo 32, so that the row
// passes' Hermitian loops (lane q on line q mod lines, element q / lines)
// spread a wave over distinct banks.
constexpr int line_stride(int elems, int lines) {
  if (lines <= 1) return elems;
  const int target = (32 + lines - 1) / lines % 32;
  return elems + (((target - elems) % 32) + 32) % 32;
}

template <int L_, int E_, int LPW_, class Fwd_, class Inv_, int LPWC_ = LPW_,
          bool ZA_ = true>
struct TPlan {
  static constexpr int L = L_, E = E_, LPW = LPW_, T = L_ / E_;
  static constexpr int NT = LPW_ * (L_ / E_);
  static constexpr int LPWC = LPWC_;
  static constexpr int NTC = LPWC_ * (L_ / E_);
  static constexpr int NTCL = (NTC + 63) / 64 * 64;  // column-pass block
  static constexpr bool ZA = ZA_;
  using Fwd = Fwd_;
  using Inv = Inv_;
  static constexpr int TWI = ct::tw_count<Fwd_>;  // the inverse's twiddles
  static const float2* twiddles() { return ct::plan_twiddles<Fwd_, Inv_>(); }
  // LDS elements per line (padded exchanges) and line strides of the row
  // passes (LS) and the column pass (LSC)
  static constexpr int LE = LineElems<L_, Fwd_>::value > LineElems<L_, Inv_>::value
                                ? LineElems<L_, Fwd_>::value
                                : LineElems<L_, Inv_>::value;
  static constexpr int LS = line_stride(LE, LPW_);
  static constexpr int LSC = line_stride(LE, LPWC_);
  // FP16 column pass: one scale per 32 consecutive threads of a workgroup
  // (SG per workgroup); scales per slice for H columns
  static constexpr int SG = (LPWC_ * (L_ / E_) + 31) / 32;
  static constexpr int scales_per_slice(int H) {
    return (H + LPWC_ - 1) / LPWC_ * SG;
  }
};

// The scale group of element `row` of column k1 in the FP16 column pass's
// output: the 32-thread group of the workgroup thread that stored it
// (thread (k1 mod LPWC) T + row mod T; the inverse's last stage stores
// rows t + r L/R1, and T = L/R1 when E = R1).
template <class P>
__device__ __forceinline__ int col_scale_index(int s, int k1, int row, int H) {
  constexpr int T = P::T, LPWC = P::LPWC;
  const int kg = k1 / LPWC;
  const int tid = (k1 - kg * LPWC) * T + row % T;
  return (s * ((H + LPWC - 1) / LPWC) + kg) * P::SG + (tid >> 5);
}

// Wt element (column k1, row) of a slice: blocks of WT_B columns, each block
// by row pairs, a pair's columns side by side, its two rows adjacent.  A row
// pass moves 16 bytes a pair and column, so two columns make 32 adjacent ones;
// the column pass reads half of every 32.  Against whole columns (WT_B = 1):
// passes of 8 x 1454^2 fwd / cols / inv 68 / 146 / 74 -> 62 / 147 / 71 us, two
// slices of 2908^2 202 / 363 / 234 -> 165 / 370 / 191 us; 4: the column pass
// loses what the row passes gain (154 us, 8 x 1454^2).  The last block holds
// what columns are left, so the workspace has no padding.
//
// Every access of the passes is a slice's base (the same for the whole
// workgroup, in scalar registers) plus a 32-bit byte offset: as 64-bit
// addresses per lane the offsets took a fifth of the passes' vector
// instructions.
constexpr unsigned WT_B = 2;
__device__ __forceinline__ unsigned wt_at(int k1, int row, int H, int rp) {
  const unsigned k0 = (unsigned)k1 / WT_B * WT_B, r = row;
  const unsigned w = min(WT_B, (unsigned)H - k0);
  return k0 * (unsigned)rp + ((r / 2) * w + ((unsigned)k1 - k0)) * 2 + r % 2;
}
// element i of a uniform base
template <typename T>
__device__ __forceinline__ T& at32(T* base, unsigned i) {
  return *reinterpret_cast<T*>(reinterpret_cast<char*>(base) +
                               i * (unsigned)sizeof(T));
}
template <typename T>
__device__ __forceinline__ const T& at32(const T* base, unsigned i) {
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) +
                                     i * (unsigned)sizeof(T));
}

// Line-search commit fused into passes A and C (CM = 0: none; 1: y = sol;
// 2: y = sol + beta (sol - xp)).  Pointers may alias (in-place update).
struct CommitPtrs {
  const float* sol;
  const float* xp;
  float* dst;
  const float* Tsol;
  const float* Tx;
  float* Tdst;
  float beta;
  float s;
};

// ---------------------------------------------------------------------------
// pass A: pair-packed forward row FFTs -> Wt
//   (+ dst = y - s x when committing a step: x is the gradient there)
// ---------------------------------------------------------------------------

// FP16 storage helpers of the mixed-precision passes
__device__ __forceinline__ unsigned pack_half2(float a, float b) {
  const __half2 h = __floats2half2_rn(a, b);
  return *reinterpret_cast<const unsigned*>(&h);
}
__device__ __forceinline__ float2 unpack_half2(unsigned u) {
  return __half22float2(*reinterpret_cast<const __half2*>(&u));
}

// Storage of the passes (HM bits): HM_IN16 the input x is FP16 with a
// per-slice power-of-two scale (x = x16 / gsc); HM_WT16 the intermediates
// Wt are FP16 (pass A output at a fixed scale, pass B output with a scale
// per 32 threads); HM_SPEC16 the spectrum is read from its FP16 copy.
// Arithmetic is FP32 throughout.  Forms used: 0 (FP32), HM_IN16 (the
// mixed-precision MBIR: FP16 gradient, FP32 spectrum and intermediates)
// and all three (the FP16-storage operator).
constexpr int HM_IN16 = 1, HM_WT16 = 2, HM_SPEC16 = 4;

template <class P, int CM, int HM>
__global__ void __launch_bounds__(P::NT)
ct_rows_fwd(const void* __restrict__ xv, void* __restrict__ wtv,
            const float2* __restrict__ tw, int n, int H, int rp, int nbps,
            CommitPtrs cp, ToeplitzHalf ha) {
  extern __shared__ float2 sm[];
  constexpr int L = P::L, E = P::E, T = P::T, LPW = P::LPW;
  using F = Xform<L, E, -1, typename P::Fwd>;
  constexpr int R1 = F::first, RS = F::last;
  const int line = threadIdx.x / T;
  const int t = threadIdx.x - line * T;
  const int b = xcd_remap(blockIdx.x, gridDim.x);
  const int s = b / nbps;
  const int r0 = (b - s * nbps) * 2 * LPW;
  const int ra = r0 + 2 * line;
  const bool hasa = ra < n, hasb = ra + 1 < n;
  // All loads first, then the commit's stores: interleaved, the compiler
  // cannot prove the stores miss later loads (dst may alias sol) and would
  // wait out each load's latency in turn.
  float2 v[E];
  float2 y[CM != 0 ? E : 1];
  const long plane = (long)s * n * n;
  const unsigned oa = (unsigned)ra * (unsigned)n;
  const float* xp = reinterpret_cast<const float*>(xv) + plane;
  const float* solp = CM != 0 ? cp.sol + plane : nullptr;
  const float* xpp = CM == 2 ? cp.xp + plane : nullptr;
  float* dstp = CM != 0 ? cp.dst + plane : nullptr;
  // FP16 input: the row-pair layout, rows ra and ra + 1 in one word
  const unsigned* xw = reinterpret_cast<const unsigned*>(xv) +
                       (long)s * ((n + 1) / 2) * n;
  const unsigned ow = (unsigned)(ra / 2) * (unsigned)n;
  static_assert(R1 % 2 == 0, "plans need an even first radix");
#pragma unroll
  for (int i = 0; i < E / R1; ++i)
#pragma unroll
    for (int r = 0; r < R1; ++r) {
      const int c = t + i * T + r * (L / R1);
      const int e = i * R1 + r;
      float re = 0.f, im = 0.f;
      if ((!P::ZA || r < R1 / 2) && c < n) {
        if constexpr ((HM & HM_IN16) != 0) {
          // the raw word (second half 0 past the last row), unpacked only
          // once every load is issued: an unpack next to its load makes
          // each load wait out its latency in turn
          if (hasa) re = __uint_as_float(at32(xw, ow + c));
        } else {
          if (hasa) re = at32(xp, oa + c);
          if (hasb) im = at32(xp, oa + n + c);
        }
        if constexpr (CM != 0) {
          float ya = 0.f, yb = 0.f;
          if (hasa) {
            ya = at32(solp, oa + c);
            if constexpr (CM == 2) ya = fmaf(cp.beta, ya - at32(xpp, oa + c), ya);
          }
          if (hasb) {
            yb = at32(solp, oa + n + c);
            if constexpr (CM == 2)
              yb = fmaf(cp.beta, yb - at32(xpp, oa + n + c), yb);
          }
          y[e] = make_float2(ya, yb);
        }
      }
      v[e] = make_float2(re, im);
    }
  if constexpr ((HM & HM_IN16) != 0) {
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = unpack_half2(__float_as_uint(v[e].x));
  }
  if constexpr (CM != 0) {
    // the step in the input's true units (FP16 input: x = g16 / gsc)
    const float se = (HM & HM_IN16) ? cp.s / ha.gsc[s] : cp.s;
#pragma unroll
    for (int i = 0; i < E / R1; ++i)
#pragma unroll
      for (int r = 0; r < (P::ZA ? R1 / 2 : R1); ++r) {
        const int c = t + i * T + r * (L / R1);
        const int e = i * R1 + r;
        if (c < n) {
          if (hasa) at32(dstp, oa + c) = fmaf(-se, v[e].x, y[e].x);
          if (hasb) at32(dstp, oa + n + c) = fmaf(-se, v[e].y, y[e].y);
        }
      }
  }
  float2* ln = sm + line * P::LS;
  F::template run<P::ZA>(v, ln, t, true, tw);
#pragma unroll
  for (int i = 0; i < E / RS; ++i)
#pragma unroll
    for (int r = 0; r < RS; ++r) ln[t + i * T + r * (L / RS)] = v[i * RS + r];
  __syncthreads();
  constexpr bool W16 = (HM & HM_WT16) != 0;
  const float hw = W16 ? 0.5f * ha.wsc : 0.5f;
  const long ws = (long)s * H * rp;  // (H rp and rows rr are even)
  for (int q = threadIdx.x; q < LPW * H; q += P::NT) {
    const int k = q / LPW;
    const int l = q - k * LPW;
    const int rr = r0 + 2 * l;
    if (rr < rp) {
      const float2 zk = sm[l * P::LS + k];
      const float2 zm = cconj(sm[l * P::LS + (k == 0 ? 0 : L - k)]);
      const float2 sp = cadd(zk, zm), df = csub(zk, zm);
      if constexpr (W16) {
        // |value| <= n * 2^16 * wsc <= 2^15: no overflow
        at32(reinterpret_cast<uint2*>(reinterpret_cast<unsigned*>(wtv) + ws),
             wt_at(k, rr, H, rp) / 2) =
            make_uint2(pack_half2(hw * sp.x, hw * sp.y),
                       pack_half2(hw * df.y, -hw * df.x));
      } else {
        at32(reinterpret_cast<float4*>(reinterpret_cast<float2*>(wtv) + ws),
             wt_at(k, rr, H, rp) / 2) =
            make_float4(hw * sp.x, hw * sp.y, hw * df.y, -hw * df.x);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// pass B: column FFT, spectrum multiply (+ spectral x.Tx), inverse FFT, all
// without leaving registers between the two transforms
// ---------------------------------------------------------------------------

template <class P, int HM>
__global__ void __launch_bounds__(P::NTCL)
ct_cols(void* __restrict__ wtv, const void* __restrict__ specv,
        const float2* __restrict__ tw, int n, int H, int rp, int nbps,
        double* partials, ToeplitzHalf ha) {
  extern __shared__ float2 sm[];
  __shared__ double red[16];
  constexpr int L = P::L, E = P::E, T = P::T, LPW = P::LPWC;
  using F = Xform<L, E, -1, typename P::Fwd>;
  using I = Xform<L, E, 1, typename P::Inv>;
  constexpr int R1 = F::first, RS = F::last;
  static_assert(I::first == RS && I::last == R1, "inverse must reverse radices");
  const int line = threadIdx.x / T;
  const int t = threadIdx.x - line * T;
  const int b = xcd_remap(blockIdx.x, gridDim.x);
  // slice-minor order: the workgroups that read spectrum rows k1 for every
  // slice run back to back on one XCD, so each row is fetched once into L2
  const int nslices = gridDim.x / nbps;
  const int kg = b / nslices;
  const int s = b - kg * nslices;
  const int k1 = kg * LPW + line;
  // threads past the last line (the block is rounded up to whole waves)
  // are inactive
  const bool active = line < LPW && k1 < H;
  const int kc = active ? k1 : 0;
  const long ws = (long)s * H * rp;
  // the slice's FP16 input scale (for the dot), fetched up front
  const float gsc_s = (HM & HM_IN16) ? ha.gsc[s] : 1.0f;
  float2 v[E];
#pragma unroll
  for (int i = 0; i < E / R1; ++i)
#pragma unroll
    for (int r = 0; r < R1; ++r) {
      const int idx = t + i * T + r * (L / R1);
      float2 w = make_float2(0.f, 0.f);
      if (r < R1 / 2 && active && idx < n) {
        const unsigned o = wt_at(kc, idx, H, rp);
        // FP16: the raw word, unpacked once every load is issued
        if constexpr ((HM & HM_WT16) != 0)
          w.x = __uint_as_float(
              at32(reinterpret_cast<const unsigned*>(wtv) + ws, o));
        else
          w = at32(reinterpret_cast<const float2*>(wtv) + ws, o);
      }
      v[i * R1 + r] = w;
    }
  if constexpr ((HM & HM_WT16) != 0) {
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = unpack_half2(__float_as_uint(v[e].x));
  }
  // the spectrum values this thread multiplies by, loaded up front so
  // their latency overlaps the forward transform
  // (an FP16 spectrum stays packed two to a register until its use, which
  // keeps the pass within the FP32 form's register budget)
  constexpr bool S16 = (HM & HM_SPEC16) != 0;
  float hs[S16 ? 1 : E];
  __half2 hs2[S16 ? (E + 1) / 2 : 1];
  {
    const unsigned so = (unsigned)kc * (unsigned)L;
#pragma unroll
    for (int i = 0; i < E / RS; ++i)
#pragma unroll
      for (int r = 0; r < RS; ++r) {
        const int e = i * RS + r;
        const unsigned o = so + t + i * T + r * (L / RS);
        if constexpr (S16) {
          const __half h = at32(reinterpret_cast<const __half*>(specv), o);
          if (e & 1)
            hs2[e / 2].y = h;
          else
            hs2[e / 2].x = h;
        } else {
          hs[e] = at32(reinterpret_cast<const float*>(specv), o);
        }
      }
  }
  float2* ln = sm + line * P::LSC;
  F::template run<true>(v, ln, t, active, tw);
  double acc = 0.0;
  if (active) {
    const float wgt = (k1 == 0 || 2 * k1 == L) ? 1.f : 2.f;
    float facc = 0.f;
#pragma unroll
    for (int i = 0; i < E / RS; ++i)
#pragma unroll
      for (int r = 0; r < RS; ++r) {
        const int e = i * RS + r;
        float h;
        if constexpr (S16)
          h = __half2float((e & 1) ? hs2[e / 2].y : hs2[e / 2].x);
        else
          h = hs[e];
        const float2 q = v[i * RS + r];
        facc += h * (q.x * q.x + q.y * q.y);
        v[i * RS + r] = cscale(q, h);
      }
    acc = (double)(wgt * facc);
  }
  // the inverse's first stage needs no exchange (same element set)
  I::run(v, ln, t, active, tw + P::TWI);
  if constexpr ((HM & HM_WT16) != 0) {
    // Power-of-two scale per 32 consecutive threads (a half wave): their
    // largest kept value maps below 2^14.  A shuffle reduction within the
    // half wave (the workgroup is a whole number of waves, so every lane
    // exists; inactive ones contribute 0); no LDS and no barrier.  Thread
    // t stores rows t + i T + r L/R1, i.e. the rows congruent to t mod T.
    float m = 0.f;
    if (active) {
#pragma unroll
      for (int i = 0; i < E / R1; ++i)
#pragma unroll
        for (int r = 0; r < R1 / 2; ++r) {
          const int idx = t + i * T + r * (L / R1);
          if (idx < n)
            m = fmaxf(m, fmaxf(fabsf(v[i * R1 + r].x),
                               fabsf(v[i * R1 + r].y)));
        }
    }
#pragma unroll
    for (int off = 16; off > 0; off >>= 1)
      m = fmaxf(m, __shfl_xor(m, off, 32));
    // m < 2^ex (frexp's exponent); all-zero and tiny groups keep ex >= -100
    int ex = 14;
    if (m > 0.f && m <= 3.0e38f)
      ex = max((int)((__float_as_uint(m) >> 23) & 0xff) - 126, -100);
    const float kap = __uint_as_float((unsigned)(127 + 14 - ex) << 23);
    if (active) {
#pragma unroll
      for (int i = 0; i < E / R1; ++i)
#pragma unroll
        for (int r = 0; r < R1 / 2; ++r) {
          const int idx = t + i * T + r * (L / R1);
          if (idx < n)
            at32(reinterpret_cast<unsigned*>(wtv) + ws, wt_at(kc, idx, H, rp)) =
                pack_half2(kap * v[i * R1 + r].x, kap * v[i * R1 + r].y);
        }
    }
    if ((threadIdx.x & 31) == 0 && (int)threadIdx.x < P::NTC)
      ha.cinv[((long)s * ((H + LPW - 1) / LPW) + kg) * P::SG +
              (threadIdx.x >> 5)] =
          ha.cbase * __uint_as_float((unsigned)(127 + ex - 14) << 23);
  } else if (active) {
#pragma unroll
    for (int i = 0; i < E / R1; ++i)
#pragma unroll
      for (int r = 0; r < R1 / 2; ++r) {
        const int idx = t + i * T + r * (L / R1);
        if (idx < n)
          at32(reinterpret_cast<float2*>(wtv) + ws, wt_at(kc, idx, H, rp)) =
              v[i * R1 + r];
      }
  }
  if (partials) {
    if constexpr (HM != 0) {
      // back to the input's true units (input scale, spectrum and Wt
      // scales folded into pconst)
      acc *= (double)ha.pconst / ((double)gsc_s * gsc_s);
    }
    double tot = block_sum(acc, red);
    if (threadIdx.x == 0) partials[b] = tot;
  }
}

// ---------------------------------------------------------------------------
// pass C: Hermitian completion, pair-packed inverse row FFTs, crop, epilogue
//   MODE 0: out = T x;  1: out = T x - b;
//   2 / 3: out = Ty - s T x with Ty = Tsol (2) or Tsol + beta (Tsol - Tx) (3)
// ---------------------------------------------------------------------------

template <class P, int MODE, int HM>
__global__ void __launch_bounds__(P::NT)
ct_rows_inv(const void* __restrict__ wtv, const float* bvec, float* out,
            const float2* __restrict__ tw, int n, int H, int rp, int nbps,
            CommitPtrs cp, ToeplitzHalf ha) {
  extern __shared__ float2 sm[];
  constexpr int L = P::L, E = P::E, T = P::T, LPW = P::LPW;
  using I = Xform<L, E, 1, typename P::Inv>;
  constexpr int R1 = I::first, RS = I::last;
  const int line = threadIdx.x / T;
  const int t = threadIdx.x - line * T;
  const int b = xcd_remap(blockIdx.x, gridDim.x);
  const int s = b / nbps;
  const int r0 = (b - s * nbps) * 2 * LPW;
  // the slice's FP16 input scale, fetched now so that its latency overlaps
  // the transform instead of delaying the epilogue
  const float gsc_s = (HM & HM_IN16) ? ha.gsc[s] : 1.0f;
  // every Wt load of the thread in flight at once, then the LDS writes
  const long ws = (long)s * H * rp;
  constexpr int HC = L / 2 + 1;
  constexpr int NQ = (LPW * HC + P::NT - 1) / P::NT;
  float4 w4[NQ];
  constexpr bool W16 = (HM & HM_WT16) != 0;
  float cs[W16 ? NQ : 1], cs1[W16 ? NQ : 1];
  // FP16 Wt: raw words, unpacked after every load is issued
  uint2 u16[W16 ? NQ : 1];
#pragma unroll
  for (int j = 0; j < NQ; ++j) {
    const int q = threadIdx.x + j * P::NT;
    const int k = q / LPW;
    const int rr = r0 + 2 * (q - k * LPW);
    w4[j] = make_float4(0.f, 0.f, 0.f, 0.f);
    if constexpr (W16) {
      cs[j] = cs1[j] = 0.f;
      u16[j] = make_uint2(0u, 0u);
    }
    if (q < LPW * H && rr < rp) {
      const unsigned o = wt_at(k, rr, H, rp) / 2;
      if constexpr (W16) {
        u16[j] = at32(reinterpret_cast<const uint2*>(
                          reinterpret_cast<const unsigned*>(wtv) + ws), o);
        // rows rr and rr + 1 may lie in different scale groups (odd T)
        const int i0 = col_scale_index<P>(s, k, rr, H);
        const int i1 = col_scale_index<P>(s, k, rr + 1, H);
        cs[j] = ha.cinv[i0];
        cs1[j] = i1 == i0 ? cs[j] : ha.cinv[i1];
      } else {
        w4[j] = at32(reinterpret_cast<const float4*>(
                         reinterpret_cast<const float2*>(wtv) + ws), o);
      }
    }
  }
  if constexpr (W16) {
#pragma unroll
    for (int j = 0; j < NQ; ++j) {
      const float2 a = unpack_half2(u16[j].x), c = unpack_half2(u16[j].y);
      w4[j] = make_float4(a.x, a.y, c.x, c.y);
    }
  }
#pragma unroll
  for (int j = 0; j < NQ; ++j) {
    const int q = threadIdx.x + j * P::NT;
    if (q < LPW * H) {
      const int k = q / LPW;
      const int l = q - k * LPW;
      float4 w = w4[j];
      if constexpr (W16) {
        w.x *= cs[j];
        w.y *= cs[j];
        w.z *= cs1[j];
        w.w *= cs1[j];
      }
      if (k == 0 || 2 * k == L) {
        w.y = 0.f;
        w.w = 0.f;
      }
      sm[l * P::LS + k] = make_float2(w.x - w.w, w.y + w.z);
      if (k > 0 && L - k >= H)
        sm[l * P::LS + L - k] = make_float2(w.x + w.w, w.z - w.y);
    }
  }
  __syncthreads();
  float2* ln = sm + line * P::LS;
  float2 v[E];
#pragma unroll
  for (int i = 0; i < E / R1; ++i)
#pragma unroll
    for (int r = 0; r < R1; ++r) v[i * R1 + r] = ln[t + i * T + r * (L / R1)];
  __syncthreads();
  I::run(v, ln, t, true, tw + P::TWI);
  const int ra = r0 + 2 * line;
  const long plane = (long)s * n * n;
  const unsigned oa = (unsigned)ra * (unsigned)n;
  float* outp = out + plane;
  const bool hasa = ra < n, hasb = ra + 1 < n;
  // FP16 input: the transform is in units of gsc times the true values;
  // an FP16 spectrum with FP32 intermediates leaves its 2^e scale here
  // (with FP16 intermediates pass B's scales include it)
  float gi = (HM & HM_IN16) ? 1.0f / gsc_s : 1.0f;
  if constexpr ((HM & HM_SPEC16) != 0 && !W16) gi *= ha.sinv;
  // Epilogue in NB batches: each batch's operands (b, or T sol and T x) are
  // all loaded before its stores, which the compiler could not otherwise
  // move past (out may alias Tsol).  Two batches instead of one take the
  // 2916-point MODE 2 kernel from 138 to 107 VGPRs, so two workgroups fit
  // on a CU: 16 % faster at 32 x 1454^2.  (Issuing the loads before the
  // transform measured slower: more registers.)
  constexpr int NB = 2, EB = E / NB;
  static_assert(E % NB == 0, "epilogue batches must divide E");
  static_assert(RS % 2 == 0, "plans need an even last inverse radix");
  const float se = (MODE >= 2 ? cp.s : 1.0f) * gi;
#pragma unroll
  for (int h = 0; h < NB; ++h) {
    float2 e0[MODE != 0 ? EB : 1], e1[MODE == 3 ? EB : 1];
    if constexpr (MODE != 0) {
      const float* src0 = (MODE == 1 ? bvec : cp.Tsol) + plane;
      const float* src1 = MODE == 3 ? cp.Tx + plane : nullptr;
#pragma unroll
      for (int j = 0; j < EB; ++j) {
        const int e = h * EB + j, i = e / RS, r = e - i * RS;
        const int c = t + i * T + r * (L / RS);
        float2 p0 = make_float2(0.f, 0.f), p1 = p0;
        if (r < RS / 2 && c < n) {
          if (hasa) p0.x = at32(src0, oa + c);
          if (hasb) p0.y = at32(src0, oa + n + c);
          if constexpr (MODE == 3) {
            if (hasa) p1.x = at32(src1, oa + c);
            if (hasb) p1.y = at32(src1, oa + n + c);
          }
        }
        e0[j] = p0;
        if constexpr (MODE == 3) e1[j] = p1;
      }
    }
#pragma unroll
    for (int j = 0; j < EB; ++j) {
      const int e = h * EB + j, i = e / RS, r = e - i * RS;
      const int c = t + i * T + r * (L / RS);
      if (r < RS / 2 && c < n) {
        const float2 q = v[e];
        float2 o = q;
        if constexpr (MODE == 0) {
          if constexpr (HM != 0) {
            o.x = q.x * gi;
            o.y = q.y * gi;
          }
        } else if constexpr (MODE == 1) {
          o.x = fmaf(q.x, gi, -e0[j].x);
          o.y = fmaf(q.y, gi, -e0[j].y);
        } else {
          float2 ty = e0[j];
          if constexpr (MODE == 3) {
            ty.x = fmaf(cp.beta, ty.x - e1[j].x, ty.x);
            ty.y = fmaf(cp.beta, ty.y - e1[j].y, ty.y);
          }
          o.x = fmaf(-se, q.x, ty.x);
          o.y = fmaf(-se, q.y, ty.y);
        }
        if (hasa) at32(outp, oa + c) = o.x;
        if (hasb) at32(outp, oa + n + c) = o.y;
      }
    }
  }
}

template <class P, int HM>
static void run_ct(const void* x, const float* b, float* out, void* wt,
                   const void* spec, int n, int H, int rp, int nslices,
                   int mode, double* partials, hipStream_t stream0,
                   double img_b, double spec_b, const Psf::StepCommit* sc,
                   const ToeplitzHalf* half, const ToeplitzStreams* ts,
                   int group_cap) {
  const float2* tw = P::twiddles();
  // kernel-timer classes: the FP16-storage passes are timed apart
  constexpr bool H16 = HM != 0;  // any FP16 storage: timed apart
  constexpr bool W16 = (HM & HM_WT16) != 0;
  const int kc_fwd = H16 ? KC_TOEPLITZ_ROWS_FWD_F16 : KC_TOEPLITZ_ROWS_FWD;
  const int kc_cols = H16 ? KC_TOEPLITZ_COLS_F16 : KC_TOEPLITZ_COLS;
  const int kc_inv = H16 ? KC_TOEPLITZ_ROWS_INV_F16 : KC_TOEPLITZ_ROWS_INV;
  const size_t smem = sizeof(float2) * P::LPW * P::LS;
  const size_t smemc = sizeof(float2) * P::LPWC * P::LSC;
  const int npairs = (n + 1) / 2;
  const int nbr = (int)cdiv(npairs, P::LPW);  // row-pass blocks per slice
  const int nbc = (int)cdiv(H, P::LPWC);      // column-pass blocks per slice
  const long img = (long)n * n;
  const int cm = sc ? (sc->xp ? 2 : 1) : 0;
  const int em = cm ? cm + 1 : mode;  // epilogue mode of pass C
  int group = toeplitz_group_slices(nslices, H, rp, W16 ? 4 : 8);
  if (group_cap > 0) group = std::min(group, group_cap);
  // per-slice algorithmic bytes (FP16 storage: the input and the
  // intermediates at half width)
  const double ib = img_b / nslices, sb = spec_b / nslices;
  const double ibx = (HM & HM_IN16) ? 0.5 * ib : ib;
  const double sbw = W16 ? 0.5 * sb : sb;
  const size_t xel = (HM & HM_IN16) ? 2 : 4;
  // streams in use: group gi runs on stream gi % nst (0: the caller's) with
  // workspace slab gi % nst.  Slab k is first used by group k, so a full
  // group on it implies (k + 1) * group <= nslices: the slabs fit in the
  // nslices-slice workspace.
  const int nst = ts == nullptr
                      ? 1
                      : std::max(1, std::min(ts->n, (int)cdiv(nslices, group)));
  if (nst > 1) {
    TC_HIP(hipEventRecord(ts->start, stream0));
    for (int k = 0; k < nst - 1; ++k)
      TC_HIP(hipStreamWaitEvent(ts->aux[k], ts->start, 0));
  }
  const long wslab = (long)group * H * rp;  // workspace elements per group
  for (int s0 = 0, gi = 0; s0 < nslices; s0 += group, ++gi) {
    const int ns = std::min(group, nslices - s0);
    const long o = (long)s0 * img;
    const int k = gi % nst;
    hipStream_t stream = k ? ts->aux[k - 1] : stream0;
    void* wtg = static_cast<char*>(wt) + (long)k * wslab * (W16 ? 4 : 8);
    CommitPtrs cp{};
    if (sc)
      cp = CommitPtrs{sc->sol + o, sc->xp ? sc->xp + o : nullptr,
                      sc->dst + o, sc->Tsol + o,
                      sc->Tx ? sc->Tx + o : nullptr, sc->Tdst + o, sc->beta,
                      sc->s};
    ToeplitzHalf ha{};
    if (half) {
      ha = *half;
      ha.gsc = half->gsc + s0;
      ha.cinv = half->cinv + (long)k * group * P::scales_per_slice(H);
    }
    const void* xg = static_cast<const char*>(x) + xel * o;
    const float* bg = b ? b + o : nullptr;
    float* og = (sc ? sc->Tdst : out) + o;
    {
      ktimer_begin(kc_fwd, stream);
      auto launch = [&](auto k) {
        allow_lds((const void*)k, smem);
        hipLaunchKernelGGL(k, dim3(nbr * ns), dim3(P::NT), smem, stream, xg,
                           wtg, tw, n, H, rp, nbr, cp, ha);
      };
      if (cm == 0) launch(ct_rows_fwd<P, 0, HM>);
      else if (cm == 1) launch(ct_rows_fwd<P, 1, HM>);
      else launch(ct_rows_fwd<P, 2, HM>);
      TC_HIP(hipGetLastError());
      // g in, Wt out; committing: sol (and xp) in, dst out
      ktimer_end(kc_fwd, stream,
                 ns * (ibx + sbw + (cm ? (cm == 2 ? 3.0 : 2.0) * ib : 0.0)));
    }
    {
      auto k = ct_cols<P, HM>;
      allow_lds((const void*)k, smemc);
      ktimer_begin(kc_cols, stream);
      hipLaunchKernelGGL(k, dim3(nbc * ns), dim3(P::NTCL), smemc, stream, wtg,
                         spec, tw, n, H, rp, nbc,
                         partials ? partials + (long)s0 * nbc : nullptr, ha);
      TC_HIP(hipGetLastError());
      // Wt in and out; the spectrum is read once per group
      ktimer_end(kc_cols, stream,
                 ns * 2.0 * sbw +
                     ((HM & HM_SPEC16) ? 2.0 : 4.0) * (double)H * P::L);
    }
    {
      ktimer_begin(kc_inv, stream);
      auto launch = [&](auto k) {
        allow_lds((const void*)k, smem);
        hipLaunchKernelGGL(k, dim3(nbr * ns), dim3(P::NT), smem, stream, wtg,
                           bg, og, tw, n, H, rp, nbr, cp, ha);
      };
      if (em == 0) launch(ct_rows_inv<P, 0, HM>);
      else if (em == 1) launch(ct_rows_inv<P, 1, HM>);
      else if (em == 2) launch(ct_rows_inv<P, 2, HM>);
      else launch(ct_rows_inv<P, 3, HM>);
      TC_HIP(hipGetLastError());
      // Wt in, out written; plus b (mode 1) or Tsol (and Tx) when committing
      const double extra = em == 1 || em == 2 ? 1.0 : (em == 3 ? 2.0 : 0.0);
      ktimer_end(kc_inv, stream, ns * (sbw + ib * (1.0 + extra)));
    }
  }
  for (int k = 0; k + 1 < nst; ++k) {
    TC_HIP(hipEventRecord(ts->done[k], ts->aux[k]));
    TC_HIP(hipStreamWaitEvent(stream0, ts->done[k], 0));
  }
}

// One FP32-only plan: columns per workgroup of the column pass, and the passes
// (Psf::apply's arguments).
struct ToeplitzPlainOps {
  int M, lpwc;
  const float2* (*twiddles)();
  void (*run)(const float* x, const float* b, float* out, float2* wt,
              const float* spec, int n, int H, int rp, int nslices, int mode,
              double* partials, hipStream_t stream, double img_b,
              double spec_b, const Psf::StepCommit* sc,
              const ToeplitzStreams* ts, int group_cap);
};

template <class P>
void run_plain(const float* x, const float* b, float* out, float2* wt,
               const float* spec, int n, int H, int rp, int nslices, int mode,
               double* partials, hipStream_t stream, double img_b,
               double spec_b, const Psf::StepCommit* sc,
               const ToeplitzStreams* ts, int group_cap) {
  run_ct<P, 0>(x, b, out, wt, spec, n, H, rp, nslices, mode, partials, stream,
               img_b, spec_b, sc, nullptr, ts, group_cap);
}

// FP32-only plans, ascending.  With those of toeplitz_ct.hip the lengths are at
// most 16 % apart, and every width from 243 to 4096 has one within 1/7 of the
// smallest smooth length that it could use.
#define TC_FOR_TOEPLITZ_PLAIN_1(X) X(486) X(512) X(576) X(648) X(864) X(972)
#define TC_FOR_TOEPLITZ_PLAIN_2(X) X(1024) X(1152) X(1296) X(1536) X(1728)
#define TC_FOR_TOEPLITZ_PLAIN_3(X) X(1944) X(2048) X(2592) X(3072) X(3456)
#define TC_FOR_TOEPLITZ_PLAIN_4(X) \
  X(3888) X(4096) X(5184) X(6144) X(6912) X(7776) X(8192)
#define TC_FOR_TOEPLITZ_PLAIN(X)                            \
  TC_FOR_TOEPLITZ_PLAIN_1(X) TC_FOR_TOEPLITZ_PLAIN_2(X)     \
  TC_FOR_TOEPLITZ_PLAIN_3(X) TC_FOR_TOEPLITZ_PLAIN_4(X)
#define TC_TOEPLITZ_PLAIN_DECL(LL) extern ToeplitzPlainOps kToeplitzPlain##LL;
TC_FOR_TOEPLITZ_PLAIN(TC_TOEPLITZ_PLAIN_DECL)
#undef TC_TOEPLITZ_PLAIN_DECL

using PlainPlan486 = TPlan<486, 18, 9, Radices<18, 9, 3>,
                            Radices<3, 9, 18>, 9>;
using PlainPlan512 = TPlan<512, 8, 4, Radices<8, 8, 8>,
                            Radices<8, 8, 8>, 4>;
using PlainPlan576 = TPlan<576, 24, 10, Radices<24, 24>,
                            Radices<24, 24>, 10>;
using PlainPlan648 = TPlan<648, 18, 7, Radices<18, 18, 2>,
                            Radices<2, 18, 18>, 7>;
using PlainPlan864 = TPlan<864, 24, 7, Radices<24, 12, 3>,
                            Radices<3, 12, 24>, 7>;
using PlainPlan972 = TPlan<972, 18, 4, Radices<18, 18, 3>,
                            Radices<3, 18, 18>, 4>;
using PlainPlan1024 = TPlan<1024, 16, 4, Radices<16, 16, 4>,
                            Radices<4, 16, 16>, 4>;
using PlainPlan1152 = TPlan<1152, 24, 5, Radices<24, 24, 2>,
                            Radices<2, 24, 24>, 5>;
using PlainPlan1296 = TPlan<1296, 36, 7, Radices<36, 36>,
                            Radices<36, 36>, 7>;
using PlainPlan1536 = TPlan<1536, 24, 4, Radices<24, 8, 8>,
                            Radices<8, 8, 24>, 4>;
using PlainPlan1728 = TPlan<1728, 24, 3, Radices<24, 24, 3>,
                            Radices<3, 24, 24>, 3>;
using PlainPlan1944 = TPlan<1944, 18, 2, Radices<18, 18, 6>,
                            Radices<6, 18, 18>, 2>;
using PlainPlan2048 = TPlan<2048, 16, 2, Radices<16, 16, 8>,
                            Radices<8, 16, 16>, 2>;
using PlainPlan2592 = TPlan<2592, 36, 3, Radices<18, 12, 12>,
                            Radices<12, 12, 18>, 3>;
using PlainPlan3072 = TPlan<3072, 24, 2, Radices<24, 8, 4, 4>,
                            Radices<4, 4, 8, 24>, 2>;
using PlainPlan3456 = TPlan<3456, 24, 2, Radices<24, 24, 6>,
                            Radices<6, 24, 24>, 1>;
using PlainPlan3888 = TPlan<3888, 36, 2, Radices<18, 18, 12>,
                            Radices<12, 18, 18>, 2>;
using PlainPlan4096 = TPlan<4096, 16, 1, Radices<16, 16, 16>,
                            Radices<16, 16, 16>, 1>;
using PlainPlan5184 = TPlan<5184, 36, 1, Radices<36, 12, 12>,
                            Radices<12, 12, 36>, 1>;
using PlainPlan6144 = TPlan<6144, 24, 1, Radices<24, 8, 8, 4>,
                            Radices<4, 8, 8, 24>, 1>;
using PlainPlan6912 = TPlan<6912, 24, 1, Radices<24, 24, 12>,
                            Radices<12, 24, 24>, 1>;
using PlainPlan7776 = TPlan<7776, 36, 1, Radices<36, 18, 12>,
                            Radices<12, 18, 36>, 1>;
using PlainPlan8192 = TPlan<8192, 32, 1, Radices<32, 16, 16>,
                            Radices<16, 16, 32>, 1>;

#define TC_TOEPLITZ_PLAIN_DEF(LL)                                  \
  ToeplitzPlainOps kToeplitzPlain##LL = {LL, PlainPlan##LL::LPWC,  \
                                         PlainPlan##LL::twiddles,       \
                                         run_plain<PlainPlan##LL>};

}  // namespace tc
