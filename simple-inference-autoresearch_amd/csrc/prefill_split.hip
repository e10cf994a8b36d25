// Prefill variants 3 and 4: few query rows over many keys (a short prompt or a draft
// over a cached prefix), the key blocks split over work-groups.
#include "host_util.hpp"
#include "prefill_kernel.hpp"
#include "prefill_launch.hpp"

namespace sia {

template <int D, class T, int VAR>
static int launch_split(PrefillLaunch& L) {
  const dim3 grid((unsigned)(L.a.nqblk * L.a.nunit * L.a.nsplit)), block(PfCfg<D, VAR>::waves * 64);
  switch (rope_variant(L.a)) {
    case kRopeNone: hipLaunchKernelGGL((prefill_fwd<D, T, kRopeNone, VAR>), grid, block, 0, L.stream, L.a); break;
    case kRopeSplit16: hipLaunchKernelGGL((prefill_fwd<D, T, kRopeSplit16, VAR>), grid, block, 0, L.stream, L.a); break;
    case kRopeInter16: hipLaunchKernelGGL((prefill_fwd<D, T, kRopeInter16, VAR>), grid, block, 0, L.stream, L.a); break;
    case kRopeSplit32: hipLaunchKernelGGL((prefill_fwd<D, T, kRopeSplit32, VAR>), grid, block, 0, L.stream, L.a); break;
    default: hipLaunchKernelGGL((prefill_fwd<D, T, kRopeInter32, VAR>), grid, block, 0, L.stream, L.a); break;
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(SIA_ERR_LAUNCH, "prefill launch: %s", hipGetErrorString(e));
  constexpr int RPB = 256 / (D / 4);
  hipLaunchKernelGGL((prefill_merge<D, T>), dim3((unsigned)((L.a.nrows + RPB - 1) / RPB)), dim3(256), 0, L.stream, L.a);
  e = hipGetLastError();
  return e == hipSuccess ? SIA_OK : fail(SIA_ERR_LAUNCH, "prefill merge launch: %s", hipGetErrorString(e));
}

int launch_prefill_split(PrefillLaunch& L) {
  const bool bf = L.dtype == SIA_BF16;
  if (L.var == 3) {
    if (L.D == 64 && bf) return launch_split<64, BF16, 3>(L);
    if (L.D == 128) return bf ? launch_split<128, BF16, 3>(L) : launch_split<128, F16, 3>(L);
  } else if (L.var == 4) {
    switch (L.D) {
      case 64: if (!bf) return launch_split<64, F16, 4>(L); break;
      case 128: if (bf) return launch_split<128, BF16, 4>(L); break;
      case 256: return bf ? launch_split<256, BF16, 4>(L) : launch_split<256, F16, 4>(L);
    }
  }
  return fail(SIA_ERR_LAUNCH, "prefill variant %d is not built for head_dim %d", L.var, L.D);
}

}  // namespace sia
