// Dispatch of the compile-time line transforms (fft_lines_ct.h) by length.
#include "fft_lines_ct.h"

namespace tc {

#define TC_OPS(LL) &kLineOps##LL,
static const LineOps* const kOps[] = {TC_FOR_LINE_LENGTHS(TC_OPS)};
#undef TC_OPS

static const LineOps* find_ops(int L) {
  for (const LineOps* o : kOps)
    if (o->L == L) return o;
  return nullptr;
}

bool fft_lines_ct_has(int L) { return find_ops(L) != nullptr; }

int fft_lines_ct_length(int n) {
  for (const LineOps* o : kOps)
    if (o->L >= n) return o->L;
  return 0;
}

void fft_prepare(int L) {
  const LineOps* o = fft_ct_enabled() ? find_ops(L) : nullptr;
  if (o) o->twiddles();
  else fft_length(L);
}

bool fft_lines_ct(const LineFFTArgs& a, int dir, hipStream_t stream) {
  const LineOps* o = find_ops(a.L);
  if (!o) return false;
  o->lines(a, dir, stream);
  return true;
}

bool fft_real_rows_ct(const RealRowsArgs& a, bool r2c, hipStream_t stream) {
  const LineOps* o = find_ops(a.L);
  if (!o) return false;
  o->real_rows(a, r2c, stream);
  return true;
}

bool fft_rays_ct(const RayArgs& a, bool to_half, hipStream_t stream) {
  TC_REQUIRE(a.N == a.L || 2 * a.N - 1 <= a.L, "ray DFT: length too short");
  const LineOps* o = find_ops(a.L);
  if (!o) return false;
  o->rays(a, to_half, stream);
  return true;
}

}  // namespace tc
