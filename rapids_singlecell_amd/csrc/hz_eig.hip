// libharmony_hip: leading eigenpairs of a symmetric matrix in FP64, for the
// covariance eigenproblem of the dense PCA (the reference calls cuML's /
// cuSOLVER's full eigensolver, preprocessing/_pca.py:71-330).
//
//   * hz_sym_tridiag: Householder reduction Q^T A Q = T in one cooperative
//     launch, the matrix held in registers (8 rows per workgroup);
//   * hz_tridiag_top: the largest eigenvalues of T by Sturm counts;
//   * hz_sym_back: eigenvectors of T to eigenvectors of A.
// The eigenvectors of T (inverse iteration, a few milliseconds) are the
// caller's.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "harmony_hip.h"
#include "hz_host.hpp"

namespace hz {

constexpr int kEigThreads = 512;
constexpr int kEigWaves = kEigThreads / kWave;
constexpr int kEigRows = 8;        // matrix rows per workgroup
constexpr int kEigMax = 2048;      // 256 workgroups x 8 rows
constexpr unsigned kEigSpin = 1u << 17;
constexpr long long kEigEmpty = -1;  // an exchange word that nobody has written yet

struct TriArgs {
  const double* A;  // n x n
  double* d;        // n
  double* e;        // n - 1
  double* tau;      // n
  double* V;        // n x ld: Householder vectors
  long long* xch;   // n x 2 x ld: per step A v and the next row, kEigEmpty at launch
  int* status;      // 0 at launch, 1 when a wait ran out
  int n, ld;
};

__device__ __forceinline__ void eig_publish(long long* p, double v) {
  long long b = __builtin_bit_cast(long long, v);
  if (b == kEigEmpty) b = 0x7FF8000000000000ll;  // a NaN by another name
  store_agent(p, b);
}

// Lanes whose bit M is clear: the sum of `a` over the two lanes that differ in
// that bit; the others: that of `b`.  One exchange for both (the permutations
// swap half of one register with the other half of another).
template <int M>
__device__ __forceinline__ double eig_fold(double a, double b) {
  const u32x2 x = __builtin_bit_cast(u32x2, a), y = __builtin_bit_cast(u32x2, b);
  if constexpr (M == 32) {
    const auto l = __builtin_amdgcn_permlane32_swap(x.x, y.x, false, false);
    const auto h = __builtin_amdgcn_permlane32_swap(x.y, y.y, false, false);
    return __builtin_bit_cast(double, u32x2{l[0], h[0]}) + __builtin_bit_cast(double, u32x2{l[1], h[1]});
  } else if constexpr (M == 16) {
    const auto l = __builtin_amdgcn_permlane16_swap(x.x, y.x, false, false);
    const auto h = __builtin_amdgcn_permlane16_swap(x.y, y.y, false, false);
    return __builtin_bit_cast(double, u32x2{l[0], h[0]}) + __builtin_bit_cast(double, u32x2{l[1], h[1]});
  } else {
    static_assert(M == 8, "lane bit");
    const bool up = (threadIdx.x & 8) != 0;
    const double keep = up ? b : a;
    const u32x2 send = __builtin_bit_cast(u32x2, up ? a : b);
    u32x2 got;  // rotation by 8 within 16 lanes
    got.x = (unsigned)__builtin_amdgcn_update_dpp(0, (int)send.x, 0x128, 0xF, 0xF, false);
    got.y = (unsigned)__builtin_amdgcn_update_dpp(0, (int)send.y, 0x128, 0xF, 0xF, false);
    return keep + __builtin_bit_cast(double, got);
  }
}

__device__ __forceinline__ double eig_wave_sum(double v) {
  v = sum16(v);
  v = eig_fold<16>(v, v);
  return eig_fold<32>(v, v);
}

// A's rows 8 wg .. 8 wg + 7 in registers; thread t holds columns t + 512 u.  Step
// k: the Householder vector v of column k (every workgroup computes it from
// row k), p = tau A v (own rows), one exchange of p and of row k + 1 as it is
// before this step's update, w = p - tau/2 (p.v) v, A -= v w^T + w v^T.  The
// exchange words start empty and are written once, so a reader needs no flag
// or fence: it reads until nothing is empty.
// What bounds it: that exchange and three sums over the workgroup per step; the
// matrix never leaves the registers.  A workgroup's words of p are one 64-byte
// line, only what is empty is read again, a workgroup without rows left
// leaves, and the sums over lanes use no LDS: 2000 x 2000 7.2 ms (11.9 with rows
// dealt out in turn, everything read at every try and LDS permutations; host
// LAPACK's reduction on 16 cores: 110 ms, a full eigensolution 196 ms).
template <int CPT>
__global__ __launch_bounds__(kEigThreads) void tridiag_kernel(TriArgs a) {
  __shared__ double s_v[kEigThreads * CPT], s_w[kEigThreads * CPT];
  __shared__ double s_r0[kEigWaves], s_r1[kEigWaves], s_p[kEigWaves][kEigRows];
  __shared__ double s_alpha;
  __shared__ int s_fail;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wv = tid / kWave;
  const int wg = blockIdx.x, r0 = wg * kEigRows, n = a.n, ld = a.ld;
  double A[kEigRows][CPT], x[CPT];
#pragma unroll
  for (int i = 0; i < kEigRows; ++i)
#pragma unroll
    for (int u = 0; u < CPT; ++u) {
      const int r = r0 + i, c = tid + kEigThreads * u;
      A[i][u] = (r < n && c < n) ? a.A[(long long)r * n + c] : 0.0;
    }
#pragma unroll
  for (int u = 0; u < CPT; ++u) {
    const int c = tid + kEigThreads * u;
    x[u] = (c < n) ? a.A[c] : 0.0;
  }
  if (tid == 0) s_fail = 0;
  for (int k = 0;; ++k) {
    if (wg == k / kEigRows)
#pragma unroll
      for (int u = 0; u < CPT; ++u)
        if (tid + kEigThreads * u == k) a.d[k] = x[u];
    // no rows left: nobody reads from this workgroup any more
    if (k == n - 1 || r0 + kEigRows - 1 <= k) return;
    const bool owner = wg == (k + 1) / kEigRows;
    long long* xp = a.xch + (long long)k * 2 * ld;
    long long* xr = xp + ld;
    if (owner) {
      const int own = (k + 1) % kEigRows;
#pragma unroll
      for (int i = 0; i < kEigRows; ++i)
        if (i == own)
#pragma unroll
          for (int u = 0; u < CPT; ++u) {
            const int c = tid + kEigThreads * u;
            if (c > k && c < n) eig_publish(xr + c, A[i][u]);
          }
    }
    // v: beta e1 = H x, H = I - tau v v^T, alpha and beta of opposite signs
    double ss = 0.0;
#pragma unroll
    for (int u = 0; u < CPT; ++u) {
      const int c = tid + kEigThreads * u;
      if (c > k + 1) ss = fma(x[u], x[u], ss);
      if (c == k + 1) s_alpha = x[u];
    }
    ss = eig_wave_sum(ss);
    if (lane == 0) s_r0[wv] = ss;
    __syncthreads();
    double sigma = 0.0;
#pragma unroll
    for (int w = 0; w < kEigWaves; ++w) sigma += s_r0[w];
    const double alpha = s_alpha;
    const bool flat = sigma == 0.0;
    const double beta = flat ? alpha : -copysign(sqrt(fma(alpha, alpha, sigma)), alpha);
    const double v1 = alpha - beta;
    const double tau = flat ? 0.0 : 2.0 / fma(v1, v1, sigma);
    double v[CPT];
#pragma unroll
    for (int u = 0; u < CPT; ++u) {
      const int c = tid + kEigThreads * u;
      v[u] = (flat || c <= k) ? 0.0 : (c == k + 1) ? v1 : x[u];
      s_v[c] = v[u];
    }
    // own rows of A v: eight sums folded over the lanes, 4 + 2 + 1 exchanges
    // without LDS
    double q[kEigRows];
#pragma unroll
    for (int i = 0; i < kEigRows; ++i) {
      q[i] = 0.0;
#pragma unroll
      for (int u = 0; u < CPT; ++u) q[i] = fma(A[i][u], v[u], q[i]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) q[i] = eig_fold<32>(q[i], q[i + 4]);
#pragma unroll
    for (int i = 0; i < 2; ++i) q[i] = eig_fold<16>(q[i], q[i + 2]);
    q[0] = eig_fold<8>(q[0], q[1]);
    // lane bits 5, 4, 3 now name the row; the sum over bits 2 .. 0 is left
    {
      auto add = [](double x, auto ctrl) __attribute__((always_inline)) {
        const u32x2 b = __builtin_bit_cast(u32x2, x);
        u32x2 o;
        o.x = (unsigned)__builtin_amdgcn_update_dpp(0, (int)b.x, decltype(ctrl)::value, 0xF, 0xF, false);
        o.y = (unsigned)__builtin_amdgcn_update_dpp(0, (int)b.y, decltype(ctrl)::value, 0xF, 0xF, false);
        return x + __builtin_bit_cast(double, o);
      };
      q[0] = add(q[0], std::integral_constant<int, 0xB1>{});   // lane ^ 1
      q[0] = add(q[0], std::integral_constant<int, 0x4E>{});   // lane ^ 2
      q[0] = add(q[0], std::integral_constant<int, 0x141>{});  // 7 - lane of 8
    }
    if ((lane & 7) == 0) s_p[wv][lane >> 3] = q[0];
    __syncthreads();
    if (tid < kEigRows) {
      const int r = r0 + tid;
      double p = 0.0;
#pragma unroll
      for (int w = 0; w < kEigWaves; ++w) p += s_p[w][tid];
      if (r > k && r < n) eig_publish(xp + r, tau * p);
    }
    if (owner) {
#pragma unroll
      for (int u = 0; u < CPT; ++u)
        a.V[(long long)k * ld + tid + kEigThreads * u] = v[u];
      if (tid == 0) {
        a.e[k] = beta;
        a.tau[k] = tau;
      }
    }
    // p and row k + 1 of every column that is left
    double p[CPT], row[CPT];
    {
      // only what is still empty is read again: reading everything until it is
      // complete would fill the fabric
      long long lp[CPT], lw[CPT];
#pragma unroll
      for (int u = 0; u < CPT; ++u) {
        const int c = tid + kEigThreads * u;
        lp[u] = lw[u] = (c > k && c < n) ? kEigEmpty : 0;
      }
      unsigned it = 0;
      while (true) {
        bool miss = false;
#pragma unroll
        for (int u = 0; u < CPT; ++u) {
          const int c = tid + kEigThreads * u;
          if (lp[u] == kEigEmpty) lp[u] = load_agent(xp + c);
          if (lw[u] == kEigEmpty) lw[u] = load_agent(xr + c);
        }
#pragma unroll
        for (int u = 0; u < CPT; ++u) miss |= lp[u] == kEigEmpty || lw[u] == kEigEmpty;
        if (!miss) break;
        if (++it >= kEigSpin) {
          s_fail = 1;
          break;
        }
      }
#pragma unroll
      for (int u = 0; u < CPT; ++u) {
        p[u] = __builtin_bit_cast(double, lp[u]);
        row[u] = __builtin_bit_cast(double, lw[u]);
      }
    }
    double pv = 0.0;
#pragma unroll
    for (int u = 0; u < CPT; ++u) pv = fma(p[u], v[u], pv);
    pv = eig_wave_sum(pv);
    if (lane == 0) s_r1[wv] = pv;
    __syncthreads();
    if (s_fail) {  // the same in every thread: set before the barrier only
      if (tid == 0) __hip_atomic_store(a.status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return;
    }
    double dot = 0.0;
#pragma unroll
    for (int w = 0; w < kEigWaves; ++w) dot += s_r1[w];
    const double half = 0.5 * tau * dot;
    double w[CPT];
#pragma unroll
    for (int u = 0; u < CPT; ++u) {
      w[u] = fma(-half, v[u], p[u]);
      s_w[tid + kEigThreads * u] = w[u];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kEigRows; ++i) {
      const double vr = s_v[r0 + i], wr = s_w[r0 + i];  // r0 + i < ld, a multiple of 8
#pragma unroll
      for (int u = 0; u < CPT; ++u) A[i][u] = fma(-wr, v[u], fma(-vr, w[u], A[i][u]));
    }
    const double vk = s_v[k + 1], wk = s_w[k + 1];
#pragma unroll
    for (int u = 0; u < CPT; ++u) {
      const int c = tid + kEigThreads * u;
      x[u] = (c > k && c < n) ? fma(-wk, v[u], fma(-vk, w[u], row[u])) : 0.0;
    }
  }
}

// Eigenvalue blockIdx.x (0 = the largest) of the tridiagonal (d, e): one wave
// cuts the interval into 65 per pass with 64 Sturm counts side by side.  The
// reciprocal is the hardware's with two Newton steps; its last-bit error acts
// like one in e^2.  Bound by the chain of one pivot after another (2000 rows,
// 50 eigenvalues: 0.75 ms; LAPACK's bisection on the host 18 ms).
static __global__ __launch_bounds__(kWave) void tridiag_top_kernel(const double* __restrict__ d,
                                                                   const double* __restrict__ e,
                                                                   int n, double* __restrict__ out) {
  __shared__ double s_d[kEigMax], s_e[kEigMax];  // diagonal; squared off-diagonal before it
  const int lane = threadIdx.x;
  double lo = INFINITY, hi = -INFINITY, emax = 0.0;
  for (int i = lane; i < n; i += kWave) {
    const double el = i > 0 ? e[i - 1] : 0.0, er = i + 1 < n ? e[i] : 0.0;
    const double rad = fabs(el) + fabs(er);
    s_d[i] = d[i];
    s_e[i] = el * el;
    lo = fmin(lo, d[i] - rad);
    hi = fmax(hi, d[i] + rad);
    emax = fmax(emax, el * el);
  }
  for (int m = kWave / 2; m > 0; m >>= 1) {
    lo = fmin(lo, __shfl_xor(lo, m, kWave));
    hi = fmax(hi, __shfl_xor(hi, m, kWave));
    emax = fmax(emax, __shfl_xor(emax, m, kWave));
  }
  __syncthreads();
  const double tiny = 1e-290 * fmax(1.0, emax);
  const double pad = 1e-14 * fmax(fabs(lo), fabs(hi)) + tiny;
  lo -= pad;
  hi += pad;
  const int want = n - (int)blockIdx.x;  // eigenvalues not above the one sought
  for (int pass = 0; pass < 14; ++pass) {
    const double step = (hi - lo) / 65.0;
    const double t = fma(step, (double)(lane + 1), lo);
    int below = 0;
    double q = 1.0;
#pragma unroll 4
    for (int i = 0; i < n; ++i) {
      double r = __builtin_amdgcn_rcp(q);
      r = fma(fma(-q, r, 1.0), r, r);
      r = fma(fma(-q, r, 1.0), r, r);
      q = fma(-s_e[i], r, s_d[i] - t);
      if (fabs(q) < tiny) q = -tiny;
      below += q < 0.0;
    }
    const unsigned long long enough = __ballot(below >= want);
    const int f = enough ? __builtin_ctzll(enough) : kWave;
    const double nlo = f > 0 ? fma(step, (double)f, lo) : lo;
    if (f < kWave) hi = fma(step, (double)(f + 1), lo);
    lo = nlo;
    if (hi - lo <= 4.4e-16 * fmax(fabs(lo), fabs(hi)) + tiny) break;
  }
  if (lane == 0) out[blockIdx.x] = 0.5 * (lo + hi);
}

// Row m of S (n values) becomes H_0 H_1 .. H_{n-3} S_m: one workgroup per
// vector, which it keeps in registers; the next reflectors are on their way
// (four steps ahead) while one is applied.
constexpr int kBackThreads = 256;
template <int EPT>
__global__ __launch_bounds__(kBackThreads) void sym_back_kernel(const double* __restrict__ V,
                                                                const double* __restrict__ tau,
                                                                int n, int ld,
                                                                double* __restrict__ S) {
  constexpr int NW = kBackThreads / kWave, AHEAD = 4;
  __shared__ double s_r[2][NW];
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wv = tid / kWave;
  double* row = S + (long long)blockIdx.x * n;
  double s[EPT], v[AHEAD][EPT], ta[AHEAD];
#pragma unroll
  for (int u = 0; u < EPT; ++u) {
    const int c = tid + kBackThreads * u;
    s[u] = (c < n) ? row[c] : 0.0;
  }
  auto load = [&](int k, double (&x)[EPT], double& t) __attribute__((always_inline)) {
    const int kk = max(k, 0);
    t = (k >= 0) ? tau[kk] : 0.0;
#pragma unroll
    for (int u = 0; u < EPT; ++u) x[u] = V[(long long)kk * ld + tid + kBackThreads * u];
  };
#pragma unroll
  for (int g = 0; g < AHEAD; ++g) load(n - 3 - g, v[g], ta[g]);
  for (int k0 = n - 3; k0 >= 0; k0 -= AHEAD) {
#pragma unroll
    for (int g = 0; g < AHEAD; ++g) {
      double dot = 0.0;
#pragma unroll
      for (int u = 0; u < EPT; ++u) dot = fma(v[g][u], s[u], dot);
      dot = eig_wave_sum(dot);
      if (lane == 0) s_r[g & 1][wv] = dot;
      __syncthreads();
      dot = 0.0;
#pragma unroll
      for (int w = 0; w < NW; ++w) dot += s_r[g & 1][w];
      const double f = -ta[g] * dot;
#pragma unroll
      for (int u = 0; u < EPT; ++u) s[u] = fma(f, v[g][u], s[u]);
      load(k0 - g - AHEAD, v[g], ta[g]);
    }
  }
#pragma unroll
  for (int u = 0; u < EPT; ++u) {
    const int c = tid + kBackThreads * u;
    if (c < n) row[c] = s[u];
  }
}

struct EigLayout {
  int cpt, ld, G;
  double *V, *tau;
  long long* xch;
  size_t bytes;
};

static bool eig_layout(int n, void* base, EigLayout& L) {
  if (n < 3 || n > kEigMax) return false;
  L.cpt = n <= kEigThreads ? 1 : n <= 2 * kEigThreads ? 2 : 4;
  L.ld = kEigThreads * L.cpt;
  L.G = (int)ceil_div(n, kEigRows);
  if (L.G > device_cu_count()) return false;
  Carve c(base);
  L.V = c.take<double>((size_t)n * L.ld);
  L.tau = c.take<double>(n);
  L.xch = c.take<long long>((size_t)n * 2 * L.ld);
  L.bytes = align_up(c.off, 256);
  return true;
}

static int eig_ws(int n, void* ws, size_t ws_bytes, EigLayout& L) {
  HZ_RET_IF(!eig_layout(n, nullptr, L), HZ_ERR_UNSUPPORTED, "matrices of 3 to %d rows only (%d)",
            kEigMax, n);
  HZ_RET_IF(!ws || ws_bytes < L.bytes, HZ_ERR_WORKSPACE, "workspace too small: %zu < %zu", ws_bytes,
            L.bytes);
  eig_layout(n, ws, L);
  return HZ_OK;
}

}  // namespace hz

using namespace hz;

extern "C" {

size_t hz_sym_eig_workspace_bytes(int n) {
  EigLayout L;
  return eig_layout(n, nullptr, L) ? L.bytes : 0;
}

int hz_sym_tridiag(const double* A, int n, double* d, double* e, int32_t* status, void* ws,
                   size_t ws_bytes, void* stream) {
  EigLayout L;
  HZ_TRY(eig_ws(n, ws, ws_bytes, L));
  HZ_RET_IF(!A || !d || !e || !status, HZ_ERR_ARG, "A, d, e and status are required");
  hipStream_t s = static_cast<hipStream_t>(stream);
  HZ_TRY(fill<long long>(L.xch, (long long)n * 2 * L.ld, kEigEmpty, s));
  HZ_TRY(fill<int>(status, 1, 0, s));
  TriArgs a;
  a.A = A;
  a.d = d;
  a.e = e;
  a.tau = L.tau;
  a.V = L.V;
  a.xch = L.xch;
  a.status = status;
  a.n = n;
  a.ld = L.ld;
  const void* kern = L.cpt == 1   ? reinterpret_cast<const void*>(tridiag_kernel<1>)
                     : L.cpt == 2 ? reinterpret_cast<const void*>(tridiag_kernel<2>)
                                  : reinterpret_cast<const void*>(tridiag_kernel<4>);
  return chained_cooperative(s, kern, L.G, kEigThreads, &a);
}

int hz_tridiag_top(const double* d, const double* e, int n, int m, double* w, void* stream) {
  HZ_RET_IF(n < 2 || n > kEigMax, HZ_ERR_UNSUPPORTED, "matrices of 2 to %d rows only (%d)", kEigMax,
            n);
  HZ_RET_IF(m < 1 || m > n, HZ_ERR_ARG, "bad number of eigenvalues %d", m);
  HZ_RET_IF(!d || !e || !w, HZ_ERR_ARG, "d, e and w are required");
  hipLaunchKernelGGL(tridiag_top_kernel, dim3(m), dim3(kWave), 0, static_cast<hipStream_t>(stream),
                     d, e, n, w);
  HZ_LAUNCHED("tridiag_top_kernel");
  return HZ_OK;
}

int hz_sym_back(int n, int m, double* S, void* ws, size_t ws_bytes, void* stream) {
  EigLayout L;
  HZ_TRY(eig_ws(n, ws, ws_bytes, L));
  HZ_RET_IF(m < 1 || m > n || !S, HZ_ERR_ARG, "bad argument");
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (L.cpt) {
    case 1: hipLaunchKernelGGL(sym_back_kernel<2>, dim3(m), dim3(kBackThreads), 0, s, L.V, L.tau, n, L.ld, S); break;
    case 2: hipLaunchKernelGGL(sym_back_kernel<4>, dim3(m), dim3(kBackThreads), 0, s, L.V, L.tau, n, L.ld, S); break;
    default: hipLaunchKernelGGL(sym_back_kernel<8>, dim3(m), dim3(kBackThreads), 0, s, L.V, L.tau, n, L.ld, S); break;
  }
  HZ_LAUNCHED("sym_back_kernel");
  return HZ_OK;
}

}  // extern "C"
