// Kernel instances of the paged decode for f32 K/V (compiled separately so the
// instances build in parallel).
#include "paged_decode_kernel.hpp"

namespace ia {

namespace {
template <int D, int G>
int run_f32(const DecodeParams& p, int src, dim3 grid, hipStream_t st, int* resident) {
  switch (src) {
    case kSrcTopk:
      if (resident) return *resident = resident_wgs<D, G, KvF32, kSrcTopk>(), IA_OK;
      return launch_paged_finalize<D, G, KvF32, kSrcTopk>(p, grid, st);
    case kSrcDense:
      if (resident) return *resident = resident_wgs<D, G, KvF32, kSrcDense>(), IA_OK;
      return launch_paged_finalize<D, G, KvF32, kSrcDense>(p, grid, st);
    case kSrcLists:
      if (resident) return *resident = resident_wgs<D, G, KvF32, kSrcLists>(), IA_OK;
      return launch_paged_finalize<D, G, KvF32, kSrcLists>(p, grid, st);
    case kSrcTopkFused:
      if (resident) return *resident = resident_wgs<D, G, KvF32, kSrcTopkFused>(), IA_OK;
      return launch_paged_finalize<D, G, KvF32, kSrcTopkFused>(p, grid, st);
    case kSrcCondFused:  // (groups of 8 at D = 128 need more registers than two waves per SIMD have)
      if constexpr (G <= 4 || D == 64) {
        if (resident) return *resident = resident_wgs<D, G, KvF32, kSrcCondFused>(), IA_OK;
        return launch_paged_finalize<D, G, KvF32, kSrcCondFused>(p, grid, st);
      } else {
        return fail(IA_ERR_UNSUPPORTED, "one-launch condition call: fp32 caches with a GQA group of 8 at head_dim 128");
      }
  }
  return fail(IA_ERR_UNSUPPORTED, "unit source");
}
}  // namespace

int dispatch_f32(const DecodeParams& p, int d, int g, int src, dim3 grid, hipStream_t st, int* resident) {
#define IA_CASE(DD, GG) \
  if (d == DD && g == GG) return run_f32<DD, GG>(p, src, grid, st, resident);
  IA_CASE(128, 4) IA_CASE(128, 8) IA_CASE(128, 2) IA_CASE(128, 1)
  IA_CASE(64, 4) IA_CASE(64, 8) IA_CASE(64, 2) IA_CASE(64, 1)
#undef IA_CASE
  return fail(IA_ERR_UNSUPPORTED, "head_dim / group combination");
}

uint64_t wait_fallbacks_f32(bool reset) { return tu_wait_fallbacks(reset); }

}  // namespace ia
