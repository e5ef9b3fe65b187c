// libharmony_hip: k-means instantiations (HZ_UNIT_PREC=0: FP32, 1: FP64).
#include "hz_host.hpp"
#include "hz_kmeans.hpp"

namespace hz {

#if HZ_UNIT_PREC == 0
using KmT = float;
#else
using KmT = double;
#endif

template <int NT, int SM>
static int launch_km(const KmMArgs<KmT>& a, int grid, hipStream_t s) {
  auto kern = kmeans_mfma_kernel<KmT, NT, SM>;
  const size_t lds = km_lds<KmT>(NT, SM, a.K, a.d);
  // (the static part holds the labels)
  if (lds + 1024 > (size_t)device_lds_limit()) return HZ_ERR_UNSUPPORTED;
  HZ_TRY(prepare_lds(reinterpret_cast<const void*>(kern), lds));
  hipLaunchKernelGGL(kern, dim3(grid), dim3(kKmThreads), lds, s, a);
  HZ_LAUNCHED("kmeans_mfma_kernel");
  return HZ_OK;
}

template <int SM>
static int launch_km_sm(const KmMArgs<KmT>& a, int grid, hipStream_t s) {
  const int nt = (int)ceil_div(a.K, 16);
  if (nt <= 4) return launch_km<4, SM>(a, grid, s);
  if (nt <= 7) return launch_km<7, SM>(a, grid, s);
  return launch_km<8, SM>(a, grid, s);
}

int launch_kmeans_assign(const KmMArgs<KmT>& a, int grid, hipStream_t s) {
  if (a.K > 128) return HZ_ERR_UNSUPPORTED;
  const int sm = (int)ceil_div(a.d, 4);
  if (sm <= 4) return launch_km_sm<4>(a, grid, s);
  if (sm <= 8) return launch_km_sm<8>(a, grid, s);
  if (sm <= 13) return launch_km_sm<13>(a, grid, s);
  if (sm <= 16) return launch_km_sm<16>(a, grid, s);
  if (sm <= 25) return launch_km_sm<25>(a, grid, s);
  if (sm <= 32) return launch_km_sm<32>(a, grid, s);
  return HZ_ERR_UNSUPPORTED;
}

}  // namespace hz
