// libharmony_hip: FP64 centroid pass instantiations.
#include "hz_cent64.hpp"
#include "hz_host.hpp"

namespace hz {

template <int TT, int NU>
static int launch_c64(Cent64Args a, int* grid, int max_grid, hipStream_t s) {
  const int tiles = (int)ceil_div(a.K, 16);
  a.tg = tiles <= TT ? 1 : tiles <= 2 * TT ? 2 : 4;
  const int parts = kCent64Waves / a.tg;
  // two workgroups per CU while every wave has 64 rows or more
  const long long want = std::min<long long>(
      std::min<long long>(max_grid, 2LL * device_cu_count()), ceil_div(a.n, 64LL * parts));
  a.rows = (int)(ceil_div(ceil_div(a.n, want * parts), 8) * 8);
  *grid = (int)ceil_div(a.n, (long long)a.rows * parts);
  auto kern = centroid64_kernel<TT, NU>;
  const size_t lds = parts > 1 ? cent64_lds(TT, NU) : 0;
  HZ_TRY(prepare_lds(reinterpret_cast<const void*>(kern), lds));
  hipLaunchKernelGGL(kern, dim3(*grid), dim3(kBlock), lds, s, a);
  HZ_LAUNCHED("centroid64_kernel");
  return HZ_OK;
}

// At most 16 tiles of sums per wave (128 registers): four cluster tiles up to
// 64 columns, two up to 128.
int launch_cent64(const Cent64Args& a, int* grid, int max_grid, hipStream_t s) {
  if (a.K > 128 || a.d > 128) return HZ_ERR_UNSUPPORTED;
  switch ((int)ceil_div(a.d, 16)) {
    case 1:
    case 2: return launch_c64<4, 2>(a, grid, max_grid, s);
    case 3: return launch_c64<4, 3>(a, grid, max_grid, s);
    case 4: return launch_c64<4, 4>(a, grid, max_grid, s);
    case 5:
    case 6: return launch_c64<2, 6>(a, grid, max_grid, s);
    case 7: return launch_c64<2, 7>(a, grid, max_grid, s);
    default: return launch_c64<2, 8>(a, grid, max_grid, s);
  }
}

}  // namespace hz
