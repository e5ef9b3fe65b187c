// Centroid pass of FP64 jobs in natural cell order: Y partials = R^T Z on FP64
// matrix cores (the sum over all cells of clustering.cu:308-372's centroid
// GEMM; the natural order makes every row of R and Z contiguous).
#pragma once

#include "hz_sweep64.hpp"

namespace hz {

struct Cent64Args {
  const double* Z;
  const double* R;
  double* Ypart;  // gridDim.x x K x d
  const Ctrl* ctrl;
  int n, d, K;
  int tg;    // wave groups along the clusters: 1, 2 or 4
  int rows;  // rows per wave, a multiple of 8
};

constexpr int kCent64Waves = kBlock / kWave;

__host__ __device__ constexpr size_t cent64_lds(int TT, int NU) {
  return (size_t)TT * NU * 4 * kWave * sizeof(double);
}

// A workgroup's four waves are tg groups of TT cluster tiles and 4 / tg parts
// of its rows; a wave keeps TT x NU tiles of 16 x 16 sums in registers and
// feeds them straight from memory: a 16-lane group of an operand is 128
// contiguous bytes of a row, the next eight rows' operands are on their way
// while these are multiplied.  The parts of the rows meet in LDS at the end.
// 1.3M cells x 100 clusters x 50 PCs: 417 us, 3.7 TB/s beside the old-row sums
// (649 us with products and sums on vector units from LDS tiles).  Bound by HBM,
// which the two share; alone by the FP64 matrix pipes, 79% busy (the tiles are
// padded to 128 x 64).  37k x 100 x 100: 31 us (92).
template <int TT, int NU>
__global__ __launch_bounds__(kBlock, 2) void centroid64_kernel(Cent64Args a) {
  extern __shared__ __align__(16) double cent64_smem[];
  if (a.ctrl->done) return;
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int lr = lane & 15, lg = lane >> 4;
  const int n = a.n, d = a.d, K = a.K;
  const int t0 = (wv % a.tg) * TT, parts = kCent64Waves / a.tg, part = wv / a.tg;
  const long long r0 = ((long long)blockIdx.x * parts + part) * a.rows;
  const int rows = (int)max(0LL, min((long long)a.rows, n - r0));

  int ko[TT], co[NU];  // columns past the end read the last one and are not written
#pragma unroll
  for (int j = 0; j < TT; ++j) ko[j] = min(16 * (t0 + j) + lr, K - 1);
#pragma unroll
  for (int i = 0; i < NU; ++i) co[i] = min(16 * i + lr, d - 1);
  doublex4 acc[TT][NU];
#pragma unroll
  for (int j = 0; j < TT; ++j)
#pragma unroll
    for (int i = 0; i < NU; ++i) acc[j][i] = doublex4{0.0, 0.0, 0.0, 0.0};

  const double* Rb = a.R + r0 * K;
  const double* Zb = a.Z + r0 * d;
  struct Step {  // eight rows: two products per tile
    double r[2][TT], z[2][NU];
  };
  // rows past the part's end: the last row again, times zero
  auto load = [&](Step& s, int row) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int q = min(row + 4 * h + lg, rows - 1);
      const double* rp = Rb + (long long)q * K;
      const double* zp = Zb + (long long)q * d;
#pragma unroll
      for (int j = 0; j < TT; ++j) s.r[h][j] = rp[ko[j]];
#pragma unroll
      for (int i = 0; i < NU; ++i) s.z[h][i] = zp[co[i]];
    }
  };
  auto multiply = [&](const Step& s, int row) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const bool ok = row + 4 * h + lg < rows;
#pragma unroll
      for (int j = 0; j < TT; ++j) {
        const double r = ok ? s.r[h][j] : 0.0;
#pragma unroll
        for (int i = 0; i < NU; ++i) acc[j][i] = mfma_f64(r, ok ? s.z[h][i] : 0.0, acc[j][i]);
      }
    }
  };
  if (rows > 0) {
    Step s0, s1;
    load(s0, 0);
    for (int row = 0; row < rows; row += 16) {
      load(s1, row + 8);
      __builtin_amdgcn_sched_barrier(0);
      multiply(s0, row);
      __builtin_amdgcn_sched_barrier(0);
      load(s0, row + 16);
      __builtin_amdgcn_sched_barrier(0);
      multiply(s1, row + 8);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // parts 1, 2, .. in turn into part 0's sums, one group of tiles at a time
  for (int p = 1; p < parts; ++p)
    for (int t = 0; t < a.tg; ++t) {
      __syncthreads();
      if (wv == p * a.tg + t)
#pragma unroll
        for (int j = 0; j < TT; ++j)
#pragma unroll
          for (int i = 0; i < NU; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) cent64_smem[((j * NU + i) * 4 + r) * kWave + lane] = acc[j][i][r];
      __syncthreads();
      if (wv == t)
#pragma unroll
        for (int j = 0; j < TT; ++j)
#pragma unroll
          for (int i = 0; i < NU; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[j][i][r] += cent64_smem[((j * NU + i) * 4 + r) * kWave + lane];
    }
  if (part != 0) return;
  double* out = a.Ypart + (long long)blockIdx.x * K * d;
#pragma unroll
  for (int j = 0; j < TT; ++j)
#pragma unroll
    for (int i = 0; i < NU; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int k = 16 * (t0 + j) + 4 * r + lg, c = 16 * i + lr;
        if (k < K && c < d) out[(long long)k * d + c] = acc[j][i][r];
      }
}

}  // namespace hz
