// Toeplitz passes of the compile-time plans with mixed-precision forms, and
// the dispatch over all plans.
#include <cstdlib>
#include <map>
#include <mutex>
#include <tuple>

#include "toeplitz_ct.h"

namespace tc {

using Plan750 = TPlan<750, 30, 10, Radices<10, 15, 5>, Radices<5, 15, 10>>;
using Plan1458 = TPlan<1458, 18, 3, Radices<18, 9, 9>, Radices<9, 9, 18>>;
using Plan2250 = TPlan<2250, 30, 3, Radices<10, 15, 15>, Radices<15, 15, 10>>;
#ifndef TC_P2916_E
#define TC_P2916_E 18
#endif
#ifndef TC_P2916_LPW
#define TC_P2916_LPW 3
#endif
#ifndef TC_P2916_LPWC
#define TC_P2916_LPWC 1
#endif
// Column pass: one column per workgroup measured 5 % faster than three at
// this length; at 2250 three per workgroup stay 20 % faster than one.
// Pass A without the zero-padding shortcut: with it, 32 x 1454^2 measured
// 8 % slower in pass A (at 5832 the shortcut is 3 % faster).
using Plan2916 = TPlan<2916, TC_P2916_E, TC_P2916_LPW, Radices<18, 18, 9>,
                       Radices<9, 18, 18>, TC_P2916_LPWC, false>;
using Plan4500 = TPlan<4500, 30, 2, Radices<10, 15, 30>, Radices<30, 15, 10>>;
using Plan4608 = TPlan<4608, 24, 2, Radices<24, 24, 8>, Radices<8, 24, 24>, 1>;
using Plan2304 = TPlan<2304, 24, 2, Radices<24, 24, 4>, Radices<4, 24, 24>, 2>;
using Plan768 = TPlan<768, 24, 6, Radices<24, 8, 4>, Radices<4, 8, 24>, 6>;
#ifndef TC_P5832_LPW
#define TC_P5832_LPW 1
#endif
using Plan5832 = TPlan<5832, 18, TC_P5832_LPW, Radices<18, 18, 18>,
                       Radices<18, 18, 18>, 1>;

// the 144 MB rule below
int toeplitz_rule_group(int nslices, int H, int rp, int elem_bytes) {
  const double per = (double)elem_bytes * H * rp;
  const int g = (int)std::max(1.0, std::floor(144e6 / per));
  return std::min(g, nslices);
}

// Group sizes picked by the autotuner (Psf::tune_groups), keyed by
// (device, H, rp, element bytes, slices).
static std::mutex g_group_mu;
static std::map<std::tuple<int, int, int, int, int>, int> g_group_tuned;

static std::tuple<int, int, int, int, int> group_key(int H, int rp,
                                                     int elem_bytes,
                                                     int nslices) {
  int dev = 0;
  TC_HIP(hipGetDevice(&dev));
  return std::make_tuple(dev, H, rp, elem_bytes, nslices);
}

// group <= 0 forgets the entry
void toeplitz_set_group(int H, int rp, int elem_bytes, int nslices,
                        int group) {
  std::lock_guard<std::mutex> lk(g_group_mu);
  const auto key = group_key(H, rp, elem_bytes, nslices);
  if (group > 0)
    g_group_tuned[key] = group;
  else
    g_group_tuned.erase(key);
}

bool toeplitz_group_tuned(int H, int rp, int elem_bytes, int nslices) {
  std::lock_guard<std::mutex> lk(g_group_mu);
  return g_group_tuned.count(group_key(H, rp, elem_bytes, nslices)) != 0;
}

// Streams for the passes (1 or 2), keyed like the group sizes.
static std::map<std::tuple<int, int, int, int, int>, int> g_streams_tuned;

void toeplitz_set_streams(int H, int rp, int elem_bytes, int nslices,
                          int streams) {
  std::lock_guard<std::mutex> lk(g_group_mu);
  const auto key = group_key(H, rp, elem_bytes, nslices);
  if (streams > 0)
    g_streams_tuned[key] = streams;
  else
    g_streams_tuned.erase(key);
}

// TOMOCAM_HIP_TOEPLITZ_STREAMS (1 .. kMaxToeplitzStreams), else the
// tuner's choice, else 1
int toeplitz_streams(int H, int rp, int elem_bytes, int nslices) {
  const char* e = std::getenv("TOMOCAM_HIP_TOEPLITZ_STREAMS");
  if (e) return std::max(1, std::min(std::atoi(e), kMaxToeplitzStreams));
  std::lock_guard<std::mutex> lk(g_group_mu);
  auto it = g_streams_tuned.find(group_key(H, rp, elem_bytes, nslices));
  return it != g_streams_tuned.end() ? it->second : 1;
}

// Slices per group of passes.  A group's Wt intermediate stays resident in
// the memory-side cache between the three passes; about 144 MB per group
// (8 slices of 1454^2 in FP32) measured 14 % faster at 32 x 1454^2 than one
// group of all slices.  Order of precedence: TOMOCAM_HIP_TOEPLITZ_SLICES
// (0: all), the autotuner's choice for this shape, the 144 MB rule.
int toeplitz_group_slices(int nslices, int H, int rp, int elem_bytes) {
  const char* e = std::getenv("TOMOCAM_HIP_TOEPLITZ_SLICES");
  if (e) {
    const int v = std::atoi(e);
    return v > 0 ? std::min(v, nslices) : nslices;
  }
  {
    std::lock_guard<std::mutex> lk(g_group_mu);
    auto it = g_group_tuned.find(group_key(H, rp, elem_bytes, nslices));
    if (it != g_group_tuned.end()) return std::min(it->second, nslices);
  }
  return toeplitz_rule_group(nslices, H, rp, elem_bytes);
}

// Slices per group for the FP16-storage passes (sizes the pass-B scale
// buffer).
int toeplitz_half_group(int nslices, int H, int rp) {
  return toeplitz_group_slices(nslices, H, rp, 4);
}

// FFT lengths with compile-time plans, ascending
extern const int kToeplitzCtSizes[] = {750, 768, 1458, 2250, 2304, 2916,
                                       4500, 4608, 5832};
// relative time per point of each plan, where two can serve one width:
// the 10 * 15 * 30 plan for 4500 (radix-5 factors, 168 VGPRs in the column
// pass) measured 1.54x the 24 * 24 * 8 plan for 4608 per point at n = 2180
// (column pass 11.7 against 7.8 ms over 20 iterations); the 10 * 15 * 15
// plan for 2250 measured 1.17x the 24 * 24 * 4 plan for 2304 at n = 1090
// (3.87 against 3.39 ms); the 10 * 15 * 5 plan for 750 1.22x the 24 * 8 * 4
// plan for 768 at n = 362 (the three passes 2.98 against 2.49 ms)
extern const float kToeplitzCtCost[] = {1.22f, 1.f,  1.f, 1.17f, 1.f,
                                        1.f,   1.54f, 1.f, 1.f};
extern const int kToeplitzCtCount = 9;

#define TC_PLAIN(LL) &kToeplitzPlain##LL,
static const ToeplitzPlainOps* const kPlain[] = {
    TC_FOR_TOEPLITZ_PLAIN(TC_PLAIN)};
#undef TC_PLAIN

static const ToeplitzPlainOps* find_plain(int M) {
  for (const ToeplitzPlainOps* o : kPlain)
    if (o->M == M) return o;
  return nullptr;
}

// the length in [m, most] with the FP32 passes, of the plans with
// mixed-precision forms and of the others, that has the least size x relative
// time (0: none)
int toeplitz_plan_length(int m, int most) {
  int best = 0;
  float best_cost = 0.f;
  auto take = [&](int M, float cost) {
    if (M < m || M > most || (best && M * cost >= best_cost)) return;
    best = M;
    best_cost = M * cost;
  };
  for (int i = 0; i < kToeplitzCtCount; ++i)
    take(kToeplitzCtSizes[i], kToeplitzCtCost[i]);
  for (const ToeplitzPlainOps* o : kPlain) take(o->M, 1.f);
  return best;
}

// column-pass lines per workgroup (0: no compile-time plan for M)
int toeplitz_ct_lpw(int M) {
  switch (M) {
    case 750: return Plan750::LPWC;
    case 1458: return Plan1458::LPWC;
    case 2250: return Plan2250::LPWC;
    case 2916: return Plan2916::LPWC;
    case 4500: return Plan4500::LPWC;
    case 4608: return Plan4608::LPWC;
    case 2304: return Plan2304::LPWC;
    case 768: return Plan768::LPWC;
    case 5832: return Plan5832::LPWC;
    default: {
      const ToeplitzPlainOps* o = find_plain(M);
      return o ? o->lpwc : 0;
    }
  }
}

// Lays out the twiddle tables of M's plan; false: no compile-time plan.
bool toeplitz_ct_prepare(int M) {
  switch (M) {
    case 750: Plan750::twiddles(); return true;
    case 1458: Plan1458::twiddles(); return true;
    case 2250: Plan2250::twiddles(); return true;
    case 2916: Plan2916::twiddles(); return true;
    case 4500: Plan4500::twiddles(); return true;
    case 4608: Plan4608::twiddles(); return true;
    case 2304: Plan2304::twiddles(); return true;
    case 768: Plan768::twiddles(); return true;
    case 5832: Plan5832::twiddles(); return true;
    default: {
      const ToeplitzPlainOps* o = find_plain(M);
      if (o) o->twiddles();
      return o != nullptr;
    }
  }
}

// FP16 column-pass scales per slice (0: no compile-time plan for M)
int toeplitz_ct_scales(int M, int H) {
  switch (M) {
    case 750: return Plan750::scales_per_slice(H);
    case 1458: return Plan1458::scales_per_slice(H);
    case 2250: return Plan2250::scales_per_slice(H);
    case 2916: return Plan2916::scales_per_slice(H);
    case 4500: return Plan4500::scales_per_slice(H);
    case 4608: return Plan4608::scales_per_slice(H);
    case 2304: return Plan2304::scales_per_slice(H);
    case 768: return Plan768::scales_per_slice(H);
    case 5832: return Plan5832::scales_per_slice(H);
    default: return 0;
  }
}

template <int HM>
static bool apply_ct(int M, const void* x, const float* b, float* out,
                     void* wt, const void* spec, int n, int H, int rp,
                     int nslices, int mode, double* partials,
                     hipStream_t stream, double img_b, double spec_b,
                     const Psf::StepCommit* sc, const ToeplitzHalf* half,
                     const ToeplitzStreams* ts, int group_cap = 0) {
#define TC_RUN_CT(PL)                                                        \
  run_ct<PL, HM>(x, b, out, wt, spec, n, H, rp, nslices, mode, partials,    \
                  stream, img_b, spec_b, sc, half, ts, group_cap);          \
  return true
  switch (M) {
    case 750: TC_RUN_CT(Plan750);
    case 1458: TC_RUN_CT(Plan1458);
    case 2250: TC_RUN_CT(Plan2250);
    case 2916: TC_RUN_CT(Plan2916);
    case 4500: TC_RUN_CT(Plan4500);
    case 4608: TC_RUN_CT(Plan4608);
    case 2304: TC_RUN_CT(Plan2304);
    case 768: TC_RUN_CT(Plan768);
    case 5832: TC_RUN_CT(Plan5832);
    default: return false;
  }
#undef TC_RUN_CT
}

bool toeplitz_apply_ct(int M, const float* x, const float* b, float* out,
                       float2* wt, const float* spec, int n, int H, int rp,
                       int nslices, int mode, double* partials,
                       hipStream_t stream, double img_b, double spec_b,
                       const Psf::StepCommit* sc, const ToeplitzStreams* ts,
                       int group_cap) {
  if (const ToeplitzPlainOps* o = find_plain(M)) {
    o->run(x, b, out, wt, spec, n, H, rp, nslices, mode, partials, stream,
           img_b, spec_b, sc, ts, group_cap);
    return true;
  }
  return apply_ct<0>(M, x, b, out, wt, spec, n, H, rp, nslices, mode,
                     partials, stream, img_b, spec_b, sc, nullptr, ts,
                     group_cap);
}

bool toeplitz_apply_ct_half(int M, const void* x16, float* out, void* wt,
                            const void* spec, int n, int H, int rp,
                            int nslices, double* partials, hipStream_t stream,
                            double img_b, double spec_b,
                            const Psf::StepCommit* sc,
                            const ToeplitzHalf& half, bool wt16,
                            const ToeplitzStreams* ts) {
  if (wt16)
    return apply_ct<HM_IN16 | HM_WT16 | HM_SPEC16>(
        M, x16, nullptr, out, wt, spec, n, H, rp, nslices, 0, partials,
        stream, img_b, spec_b, sc, &half, ts);
  return apply_ct<HM_IN16>(M, x16, nullptr, out, wt, spec, n, H, rp,
                           nslices, 0, partials, stream, img_b, spec_b, sc,
                           &half, ts);
}

}  // namespace tc
