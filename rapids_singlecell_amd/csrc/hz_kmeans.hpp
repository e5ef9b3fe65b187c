// Lloyd step of the k-means initialiser on matrix cores (the reference calls
// cuML KMeans, _harmony/__init__.py:292-353): scores z.y - |y|^2 / 2, the
// label is the largest score's cluster (the lowest of equal ones), and the
// clusters' sums are fixed point, so they do not depend on any order.
#pragma once

#include "hz_sweep64.hpp"

namespace hz {

constexpr int kKmThreads = 512;
constexpr int kKmWaves = kKmThreads / kWave;

template <typename T>
struct KmMArgs {
  const T* Z;
  const T* Y;       // K x d centroids
  long long* part;  // gridDim.x x (K d + K) fixed-point sums and counts
  int n, d, K;
  double scale;
};

// LDS row stride of the staged centroids: the four lane groups of an operand
// read cover the 64 banks.
template <typename T>
__host__ __device__ constexpr int km_stride(int NT) {
  return sizeof(T) == 8 ? sw64_stride(NT) : (16 * NT + 63) / 64 * 64 + 16;
}
template <typename T>
__host__ __device__ inline size_t km_lds(int NT, int SM, int K, int d) {
  return ((size_t)4 * SM * km_stride<T>(NT) + 16 * NT) * sizeof(T) + ((size_t)K * d + K) * 8;
}

__device__ __forceinline__ floatx4 km_mfma(float a, float b, floatx4 c) { return mfma_f32(a, b, c); }
__device__ __forceinline__ doublex4 km_mfma(double a, double b, doublex4 c) { return mfma_f64(a, b, c); }

// A wave labels 16 rows at a time (the next rows' loads in flight), then adds
// them to its workgroup's sums in LDS, reading the rows again along their
// length so that the adds fall on different banks also where neighbouring
// cells share a cluster.
// Per Lloyd step, with the reduction below: 200k cells x 50 PCs, 100 clusters,
// FP64 118 us (248 with products on vector units, a launch of one workgroup for
// the transposed centroids and one wave per reduced value); sixteen FP32 jobs of
// 2k to 60k cells 27 us on average (57).  Bound by the LDS adds and, below about
// 10k cells, by staging the centroids and writing the sums.
template <typename T, int NT, int SM>
__global__ __launch_bounds__(kKmThreads) void kmeans_mfma_kernel(KmMArgs<T> a) {
  using Acc = decltype(km_mfma(T(0), T(0), {}));
  constexpr int YS = km_stride<T>(NT);
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ int s_lab[kKmWaves][16];
  T* Ys = reinterpret_cast<T*>(smem);  // 4 SM x YS
  T* s_half = Ys + 4 * SM * YS;        // 16 NT
  unsigned long long* sums = reinterpret_cast<unsigned long long*>(s_half + 16 * NT);
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int lr = lane & 15, lg = lane >> 4;
  const int d = a.d, K = a.K, KD = K * d;
  const int tiles = (a.n + 15) / 16, step = gridDim.x * kKmWaves;
  int t = blockIdx.x * kKmWaves + wv;

  // rows 16 t + lr, columns 4 s + lg; past n or d: zero
  T za[SM];
  auto load = [&](int tile) __attribute__((always_inline)) {
    const long long row = (long long)tile * 16 + lr;
    const T* src = a.Z + (row < a.n ? row : 0) * d;
#pragma unroll
    for (int s = 0; s < SM; ++s) {
      const int c = 4 * s + lg;
      const T v = src[c < d ? c : d - 1];
      za[s] = (row < a.n && c < d) ? v : T(0);
    }
  };
  if (t < tiles) load(t);
  for (int e = tid; e < 4 * SM * YS; e += kKmThreads) Ys[e] = T(0);
  for (int e = tid; e < KD + K; e += kKmThreads) sums[e] = 0;
  __syncthreads();
  for (int e = tid; e < KD; e += kKmThreads) {
    const int k = e / d, c = e - k * d;
    Ys[c * YS + k] = a.Y[e];
  }
  __syncthreads();
  for (int k = tid; k < 16 * NT; k += kKmThreads) {
    T ss = T(0);
    for (int c = 0; c < d; ++c) ss += Ys[c * YS + k] * Ys[c * YS + k];
    s_half[k] = (k < K) ? T(0.5) * ss : T(INFINITY);
  }
  __syncthreads();
  T half[NT];
#pragma unroll
  for (int q = 0; q < NT; ++q) half[q] = s_half[16 * q + lr];

  for (; t < tiles; t += step) {
    Acc acc[NT];
#pragma unroll
    for (int q = 0; q < NT; ++q) acc[q] = Acc{T(0), T(0), T(0), T(0)};
#pragma unroll
    for (int s = 0; s < SM; ++s)
#pragma unroll
      for (int q = 0; q < NT; ++q)
        acc[q] = km_mfma(za[s], Ys[(4 * s + lg) * YS + 16 * q + lr], acc[q]);
    if (t + step < tiles) load(t + step);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      T best = -INFINITY;
      int at = 0x7fffffff;
#pragma unroll
      for (int q = 0; q < NT; ++q) {
        const T sc = acc[q][r] - half[q];
        if (sc > best) {
          best = sc;
          at = 16 * q + lr;
        }
      }
#pragma unroll
      for (int m = 8; m > 0; m >>= 1) {
        const T ob = __shfl_xor(best, m, kWave);
        const int oi = __shfl_xor(at, m, kWave);
        if (ob > best || (ob == best && oi < at)) {
          best = ob;
          at = oi;
        }
      }
      // non-finite scores: an index in range
      if (lr == 0) s_lab[wv][sizeof(T) == 8 ? 4 * r + lg : 4 * lg + r] = at < K ? at : 0;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const long long row0 = (long long)t * 16;
    const int rows = (int)min(16LL, (long long)a.n - row0);
    const T* src = a.Z + row0 * d;
    int r = lane / d, c = lane - r * d;
#pragma unroll 4
    for (int e = lane; e < rows * d; e += kWave) {
      const long long v = to_fixed((double)src[e], a.scale);
      atomicAdd(&sums[s_lab[wv][r] * d + c], (unsigned long long)v);
      for (c += kWave; c >= d; c -= d) ++r;
    }
    if (lane < rows) atomicAdd(&sums[KD + s_lab[wv][lane]], 1ull);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }
  __syncthreads();
  long long* out = a.part + (long long)blockIdx.x * (KD + K);
  for (int e = tid; e < KD + K; e += kKmThreads) out[e] = (long long)sums[e];
}

// New centroid of cluster blockIdx.x: its partial sums over their count (a
// cluster with no cells keeps its centroid).  Sixteen waves share the G
// partials, lanes the columns, sixteen loads in flight per wave.
constexpr int kKmUpdThreads = 1024;
template <typename T>
__global__ __launch_bounds__(kKmUpdThreads) void kmeans_mean_kernel(
    const long long* __restrict__ part, int G, T* __restrict__ Y, int K, int d, double inv_scale) {
  constexpr int NW = kKmUpdThreads / kWave, U = 16;
  __shared__ long long s_sum[NW][kWave], s_cnt[NW];
  const int k = blockIdx.x, lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
  const long long stride = (long long)K * d + K;
  long long cnt = 0;
  for (int g = threadIdx.x; g < G; g += kKmUpdThreads) cnt += part[g * stride + (long long)K * d + k];
#pragma unroll
  for (int m = kWave / 2; m > 0; m >>= 1) cnt += __shfl_xor(cnt, m, kWave);
  if (lane == 0) s_cnt[wv] = cnt;
  for (int c0 = 0; c0 < d; c0 += kWave) {
    const int c = min(c0 + lane, d - 1);
    const long long* src = part + (long long)k * d + c;
    long long s = 0;
    for (int g0 = wv; g0 < G; g0 += NW * U) {
      long long v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) v[u] = src[min(g0 + u * NW, G - 1) * stride];
#pragma unroll
      for (int u = 0; u < U; ++u) s += (g0 + u * NW < G) ? v[u] : 0;
    }
    __syncthreads();
    s_sum[wv][lane] = s;
    __syncthreads();
    if (wv == 0 && c0 + lane < d) {
      long long tot = 0, n = 0;
      for (int w = 0; w < NW; ++w) {
        tot += s_sum[w][lane];
        n += s_cnt[w];
      }
      if (n > 0) Y[(long long)k * d + c] = T((double)tot * inv_scale / (double)n);
    }
  }
}

}  // namespace hz
