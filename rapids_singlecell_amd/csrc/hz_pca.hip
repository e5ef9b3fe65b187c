// libharmony_hip: dense PCA producer of the Harmony input (pp.pca with
// zero_center=True): column means, the covariance of the centred matrix on
// matrix cores, and the projection onto the leading eigenvectors.
//
//   * means: per-slice FP64 column sums (coalesced along rows), reduced in
//     slice order;
//   * covariance: one workgroup per (64 x 64 or 128 x 128 upper-triangle tile,
//     row slice); strips of the centred rows are staged in LDS and multiplied
//     on v_mfma_f32_16x16x4f32 (FP32 products and accumulation within a
//     slice); the slices are summed in FP64 in slice order, divided
//     by n - 1 and mirrored;
//   * projection: one workgroup per 64 rows; centred row tiles and the
//     eigenvector tile are staged in LDS and multiplied on matrix cores.
// The leading eigenpairs of the (n_vars x n_vars) covariance are hz_eig.hip's.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "harmony_hip.h"
#include "hz_host.hpp"

namespace hz {

constexpr int kPcaT = 64;       // projection rows per workgroup, columns per step
constexpr int kPcaR = 32;       // rows staged per step of the covariance kernel
constexpr int kPcaSlices = 256;    // row slices of the moment pass

static __global__ void pca_to_float_kernel(const double* __restrict__ m, float* __restrict__ f,
                                           int g) {
  for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < g; c += gridDim.x * blockDim.x)
    f[c] = (float)m[c];
}

// Per-slice column sums (FP64); slice s covers rows [s*per, (s+1)*per).
static __global__ void pca_colsum_kernel(const float* __restrict__ X, long long n, int g,
                                         long long per, double* __restrict__ part) {
  const long long r0 = (long long)blockIdx.y * per;
  const long long r1 = min(n, r0 + per);
  for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < g; c += gridDim.x * blockDim.x) {
    double s = 0.0;
    for (long long r = r0; r < r1; ++r) s += (double)X[r * g + c];
    part[(long long)blockIdx.y * g + c] = s;
  }
}

static __global__ void pca_mean_kernel(const double* __restrict__ part, int slices, int g,
                                       long long n, double* __restrict__ mean,
                                       float* __restrict__ meanf) {
  for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < g; c += gridDim.x * blockDim.x) {
    double s = 0.0;
    for (int q = 0; q < slices; ++q) s += part[(long long)q * g + c];
    mean[c] = s / (double)n;
    meanf[c] = (float)(s / (double)n);
  }
}

// Covariance partials: workgroup (tile t, slice y) accumulates
// sum_r (x_ri - m_i)(x_rj - m_j) for the tile's E x E (i, j) block over the
// slice's rows, each wave a quarter.  Tiles enumerate the upper triangle
// (bi <= bj).  Rows stay rows in LDS: an operand read takes 16 columns of four
// rows, which the stride puts on 64 banks; the next stage's rows are on their
// way during the products.  The sum's order (slices of the rows, four rows per
// instruction) does not depend on E.
// Bound by the FP32 matrix cores: 50k x 2000 2.87 ms (5.48 when each wave
// had one 16-column A operand for four products and staged columns one value
// at a time; the products alone take 1.5 ms).  E = 128 reads LDS half as often
// per product; E = 64 where the larger tiles would leave CUs idle.
// VEC: rows are read 16 bytes at a time (n_cols % 4 == 0).
template <int E, bool VEC>
static __global__ __launch_bounds__(kBlock, 2) void pca_cov_kernel(const float* __restrict__ X,
                                                                   long long n, int g,
                                                                   const float* __restrict__ meanf,
                                                                   int nb, long long per,
                                                                   float* __restrict__ part) {
  constexpr int Q = E / 4;               // column quads of a strip
  constexpr int U = kPcaR * Q / kBlock;  // quads per thread, strip and stage
  constexpr int W = E / 2, M = W / 16;   // a wave's quarter: W columns, M operand tiles
  __shared__ __align__(16) float s_x[2][kPcaR][E + 16];
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wv = tid / kWave;
  const int lr = lane & 15, lg = lane >> 4;
  // tile index -> (bi, bj), bi <= bj
  int t = blockIdx.x, bi = 0;
  while (t >= nb - bi) {
    t -= nb - bi;
    ++bi;
  }
  const int bj = bi + t;
  const long long r0 = (long long)blockIdx.y * per;
  const long long r1 = min(n, r0 + per);
  // this thread's column quad of either strip and its means
  const int q4 = 4 * (tid % Q), rr0 = tid / Q;
  int col[2];
  float m[2][4];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    col[h] = (h ? bj : bi) * E + q4;
#pragma unroll
    for (int i = 0; i < 4; ++i) m[h][i] = (col[h] + i < g) ? meanf[col[h] + i] : 0.f;
  }
  float x[2][U][4];
  auto load = [&](long long rb) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const long long r = rb + rr0 + u * (kBlock / Q);
      const float* row = X + min(r, n - 1) * g;  // rows past the slice are masked below
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if constexpr (VEC) {
          const floatx4 v = *reinterpret_cast<const floatx4*>(row + min(col[h], g - 4));
#pragma unroll
          for (int i = 0; i < 4; ++i) x[h][u][i] = v[i];
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i) x[h][u][i] = row[min(col[h] + i, g - 1)];
        }
      }
    }
  };
  auto store = [&](long long rb) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int rr = rr0 + u * (kBlock / Q);
      const bool ok = rb + rr < r1;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        floatx4 v;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = (ok && col[h] + i < g) ? x[h][u][i] - m[h][i] : 0.f;
        *reinterpret_cast<floatx4*>(&s_x[h][rr][q4]) = v;
      }
    }
  };
  floatx4 acc[M][M];
#pragma unroll
  for (int i = 0; i < M; ++i)
#pragma unroll
    for (int j = 0; j < M; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  const int ci = W * (wv & 1) + lr, cj = W * (wv >> 1) + lr;  // this wave's quarter
  if (r0 < r1) load(r0);
  for (long long rb = r0; rb < r1; rb += kPcaR) {
    __syncthreads();
    store(rb);
    __syncthreads();
    if (rb + kPcaR < r1) load(rb + kPcaR);
    float av[2][M], bv[2][M];
    auto rd = [&](int s, int o) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < M; ++i) {
        av[o][i] = s_x[0][4 * s + lg][ci + 16 * i];
        bv[o][i] = s_x[1][4 * s + lg][cj + 16 * i];
      }
    };
    rd(0, 0);
#pragma unroll
    for (int s = 0; s < kPcaR / 4; ++s) {
      if (s + 1 < kPcaR / 4) rd(s + 1, (s + 1) & 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < M; ++i)
#pragma unroll
        for (int j = 0; j < M; ++j) acc[i][j] = mfma_f32(av[s & 1][i], bv[s & 1][j], acc[i][j]);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // D[4 lg + r][lr] of subtile (i, j)
  float* out = part + ((long long)blockIdx.y * gridDim.x + blockIdx.x) * E * E;
#pragma unroll
  for (int i = 0; i < M; ++i)
#pragma unroll
    for (int j = 0; j < M; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        out[(W * (wv & 1) + 16 * i + 4 * lg + r) * E + cj + 16 * j] = acc[i][j][r];
}

// Sum of the slices (FP64, slice order), / (n - 1), both triangles.
static __global__ void pca_cov_reduce_kernel(const float* __restrict__ part, int tiles, int slices,
                                             int nb, int edge, int g, long long n,
                                             double* __restrict__ cov) {
  const long long te = (long long)edge * edge, tot = tiles * te;
  for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < tot;
       e += (long long)gridDim.x * blockDim.x) {
    int t = (int)(e / te);
    const int w = (int)(e - t * te);
    const int ii = w / edge, jj = w - ii * edge;
    int bi = 0;
    while (t >= nb - bi) {
      t -= nb - bi;
      ++bi;
    }
    const int bj = bi + t;
    const int i = bi * edge + ii, j = bj * edge + jj;
    if (i >= g || j >= g) continue;
    double s = 0.0;
    for (int q = 0; q < slices; ++q) s += (double)part[(long long)q * tot + e];
    s /= (double)(n - 1);
    cov[(long long)i * g + j] = s;
    cov[(long long)j * g + i] = s;
  }
}

// out[r][c] = sum_i (x_ri - m_i) V[i][c], 64 rows per workgroup, nc <= 64.
static __global__ __launch_bounds__(kBlock) void pca_project_kernel(
    const float* __restrict__ X, long long n, int g, const float* __restrict__ meanf,
    const float* __restrict__ V, int nc, float* __restrict__ out) {
  __shared__ float sX[kPcaT][kPcaT + 4];  // row, column (of the 64-column strip)
  __shared__ float sV[kPcaT][kPcaT + 4];  // column of the strip, component
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wv = tid / kWave;
  const int lr = lane & 15, lg = lane >> 4;
  const long long rbase = (long long)blockIdx.x * kPcaT;
  floatx4 acc[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) acc[q] = floatx4{0.f, 0.f, 0.f, 0.f};
  for (int cb = 0; cb < g; cb += kPcaT) {
    __syncthreads();
    for (int e = tid; e < kPcaT * kPcaT; e += kBlock) {
      const int rr = e / kPcaT, cc = e - rr * kPcaT;
      const long long r = rbase + rr;
      const int c = cb + cc;
      sX[rr][cc] = (r < n && c < g) ? X[r * g + c] - meanf[c] : 0.f;
      // e also indexes (gene cc', component) for the eigenvector tile
      const int gi = e / kPcaT, comp = e - gi * kPcaT;
      sV[gi][comp] = (cb + gi < g && comp < nc) ? V[(long long)(cb + gi) * nc + comp] : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < kPcaT / 4; ++s) {
      const float av = sX[16 * wv + lr][4 * s + lg];
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[q] = mfma_f32(av, sV[4 * s + lg][16 * q + lr], acc[q]);
    }
  }
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const long long row = rbase + 16 * wv + 4 * lg + r;
      const int comp = 16 * q + lr;
      if (row < n && comp < nc) out[row * nc + comp] = acc[q][r];
    }
}

struct PcaLayout {
  int nb, tiles, slices, edge;
  long long per;
  double* colpart;
  float* meanf;
  float* covpart;
  size_t bytes;
};

static void pca_layout(long long n, int g, void* base, PcaLayout& P) {
  // enough (64 x 64 tile, slice) pairs to fill the device, slices of >= 2048
  // rows
  const int nb = (int)ceil_div(g, 64), tiles = nb * (nb + 1) / 2;
  P.slices = (int)std::max<long long>(1, std::min<long long>(ceil_div(n, 2048),
                                                            ceil_div(2048, tiles)));
  P.per = ceil_div(n, P.slices);
  const int nb2 = (int)ceil_div(g, 128);
  P.edge = nb2 * (nb2 + 1) / 2 * P.slices < 256 ? 64 : 128;
  P.nb = P.edge == 64 ? nb : nb2;
  P.tiles = P.nb * (P.nb + 1) / 2;
  Carve c(base);
  P.colpart = c.take<double>((size_t)kPcaSlices * g);
  P.meanf = c.take<float>(g);
  P.covpart = c.take<float>((size_t)P.slices * P.tiles * P.edge * P.edge);
  P.bytes = align_up(c.off, 256);
}

}  // namespace hz

using namespace hz;

extern "C" {

size_t hz_pca_workspace_bytes(long long n_rows, int n_cols) {
  if (n_rows < 2 || n_cols < 1) return 0;
  PcaLayout P;
  pca_layout(n_rows, n_cols, nullptr, P);
  return P.bytes;
}

int hz_pca_covariance(const float* X, long long n_rows, int n_cols, double* mean, double* cov,
                      void* ws, size_t ws_bytes, void* stream) {
  HZ_RET_IF(n_rows < 2 || n_cols < 1, HZ_ERR_ARG, "bad shape (n=%lld g=%d)", n_rows, n_cols);
  HZ_RET_IF(!X || !mean || !cov, HZ_ERR_ARG, "X, mean and cov are required");
  PcaLayout P;
  pca_layout(n_rows, n_cols, nullptr, P);
  HZ_RET_IF(!ws || ws_bytes < P.bytes, HZ_ERR_WORKSPACE, "workspace too small: %zu < %zu",
            ws_bytes, P.bytes);
  pca_layout(n_rows, n_cols, ws, P);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const long long per_m = (n_rows + kPcaSlices - 1) / kPcaSlices;
  hipLaunchKernelGGL(pca_colsum_kernel, dim3((n_cols + 255) / 256, kPcaSlices), dim3(256), 0, s, X,
                     n_rows, n_cols, per_m, P.colpart);
  HZ_LAUNCHED("pca_colsum_kernel");
  hipLaunchKernelGGL(pca_mean_kernel, dim3((n_cols + 255) / 256), dim3(256), 0, s, P.colpart,
                     kPcaSlices, n_cols, n_rows, mean, P.meanf);
  HZ_LAUNCHED("pca_mean_kernel");
  const bool vec = n_cols % 4 == 0 && reinterpret_cast<uintptr_t>(X) % 16 == 0;
  auto cov_kernel = P.edge == 64 ? (vec ? pca_cov_kernel<64, true> : pca_cov_kernel<64, false>)
                                 : (vec ? pca_cov_kernel<128, true> : pca_cov_kernel<128, false>);
  hipLaunchKernelGGL(cov_kernel, dim3(P.tiles, P.slices), dim3(kBlock), 0, s, X, n_rows, n_cols,
                     P.meanf, P.nb, P.per, P.covpart);
  HZ_LAUNCHED("pca_cov_kernel");
  const long long tot = (long long)P.tiles * P.edge * P.edge;
  hipLaunchKernelGGL(pca_cov_reduce_kernel, dim3((int)std::min<long long>(4096, (tot + 255) / 256)),
                     dim3(256), 0, s, P.covpart, P.tiles, P.slices, P.nb, P.edge, n_cols, n_rows, cov);
  HZ_LAUNCHED("pca_cov_reduce_kernel");
  return HZ_OK;
}

int hz_pca_project(const float* X, long long n_rows, int n_cols, const double* mean,
                   const float* components, int n_comps, float* out, void* ws, size_t ws_bytes,
                   void* stream) {
  HZ_RET_IF(n_rows < 1 || n_cols < 1 || n_comps < 1, HZ_ERR_ARG, "bad shape");
  HZ_RET_IF(n_comps > kPcaT, HZ_ERR_UNSUPPORTED, "n_comps=%d > %d is not supported", n_comps,
            kPcaT);
  HZ_RET_IF(!X || !mean || !components || !out, HZ_ERR_ARG, "null argument");
  PcaLayout P;
  pca_layout(std::max(2LL, n_rows), n_cols, nullptr, P);
  HZ_RET_IF(!ws || ws_bytes < P.bytes, HZ_ERR_WORKSPACE, "workspace too small: %zu < %zu",
            ws_bytes, P.bytes);
  pca_layout(std::max(2LL, n_rows), n_cols, ws, P);
  hipStream_t s = static_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(pca_to_float_kernel, dim3((n_cols + 255) / 256), dim3(256), 0, s, mean,
                     P.meanf, n_cols);
  HZ_LAUNCHED("pca_to_float_kernel");
  hipLaunchKernelGGL(pca_project_kernel, dim3((int)((n_rows + kPcaT - 1) / kPcaT)), dim3(kBlock),
                     0, s, X, n_rows, n_cols, P.meanf, components, n_comps, out);
  HZ_LAUNCHED("pca_project_kernel");
  return HZ_OK;
}

}  // extern "C"
