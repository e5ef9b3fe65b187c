// libharmony_hip: FP64 block sweep instantiations.
#include "hz_host.hpp"

namespace hz {

template <int NT, int SM>
static int launch_sw64(const Layout& L, const Sweep64Args* a, int* Gp, hipStream_t s) {
  auto kern = sweep64_kernel<NT, SM>;
  const size_t lds = sweep64_lds(SM, NT, L.B, L.K, L.pd.nblk);
  if (prepare_lds(reinterpret_cast<const void*>(kern), lds) != HZ_OK) return HZ_ERR_UNSUPPORTED;
  int per_cu = 0;
  HZ_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(kern),
                                                      kSw64Threads, lds));
  if (per_cu < 1) return HZ_ERR_UNSUPPORTED;
  if (!a) {
    const int cap = device_cu_count();
    *Gp = tune_value(HZ_TUNE_SWEEP_WG) > 0 ? std::min(tune_value(HZ_TUNE_SWEEP_WG), cap)
                                           : sweep_wgs(L, cap, kSw64Waves);
    return HZ_OK;
  }
  if (tune_value(HZ_TUNE_SWEEP_PLAIN)) {
    // same grid, within the co-resident capacity computed above
    hipLaunchKernelGGL(kern, dim3((unsigned)*Gp), dim3(kSw64Threads), lds, s, *a);
    HZ_LAUNCHED("sweep64_kernel");
    return HZ_OK;
  }
  void* args[] = {const_cast<Sweep64Args*>(a)};
  const hipError_t e =
      hipLaunchCooperativeKernel(reinterpret_cast<const void*>(kern), dim3((unsigned)*Gp),
                                 dim3(kSw64Threads), args, (unsigned)lds, s);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    mark_sweep_broken();
    return HZ_ERR_UNSUPPORTED;
  }
  return HZ_OK;
}

template <int SM>
static int launch_sw64_sm(const Layout& L, const Sweep64Args* a, int* G, hipStream_t s) {
  switch (L.NT) {
    case 4: return launch_sw64<4, SM>(L, a, G, s);
    case 7: return launch_sw64<7, SM>(L, a, G, s);
    case 8: return launch_sw64<8, SM>(L, a, G, s);
    default: return HZ_ERR_UNSUPPORTED;
  }
}

// a == nullptr: choose the grid only; HZ_ERR_UNSUPPORTED (nothing launched)
// when the shape has no kernel or cannot be made co-resident
int launch_sweep64(const Layout& L, const Sweep64Args* a, int* G, hipStream_t s) {
  switch (row_sm(L)) {
    case 4: return launch_sw64_sm<4>(L, a, G, s);
    case 8: return launch_sw64_sm<8>(L, a, G, s);
    case 13: return launch_sw64_sm<13>(L, a, G, s);
    case 16: return launch_sw64_sm<16>(L, a, G, s);
    case 25: return launch_sw64_sm<25>(L, a, G, s);
    default: return HZ_ERR_UNSUPPORTED;
  }
}

}  // namespace hz
