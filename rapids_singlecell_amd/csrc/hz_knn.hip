// libharmony_hip: exact k nearest neighbours (brute force) of every row of an
// embedding among all its rows -- the neighbour search that consumes the
// integrated embedding (pp.neighbors with algorithm="brute").
//
// The rows are first laid out as tiles of 64 candidates, dimension-major and
// zero padded, with a row of norms (knn_pack_kernel).  One workgroup owns 128
// query rows (8 waves x 16) and streams one part of the tiles through LDS:
//   * the query x candidate dot products run on matrix cores
//     (v_mfma_f32_16x16x4f32: FP32 products, FP32 accumulation), the queries
//     held in registers as the A operand for the whole stream;
//   * a distance (euclidean / squared euclidean from the expanded form
//     |x|^2 + |y|^2 - 2 x.y, cosine as 1 - x.y of unit rows) is compared, in
//     the registers the product left it in, with its query's threshold, the
//     k-th smallest distance known so far;
//   * the few that pass are appended to the query's buffer in LDS; a buffer
//     that may overflow is cut to its k smallest (distance, index) keys, which
//     lowers the threshold.
// The lists of the parts are merged by knn_merge_kernel.
// Distances are computed in FP32 as the reference's GPU search does
// (cuML NearestNeighbors(algorithm="brute"), _neighbors/_algorithms/_brute.py).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>

#include "harmony_hip.h"
#include "hz_host.hpp"

namespace hz {

constexpr int kKnnQ = 128;            // queries per workgroup
constexpr int kKnnThreads = kKnnQ / 16 * kWave;
constexpr int kKnnC = 64;             // candidates per tile
constexpr int kKnnCS = kKnnC + 16;    // LDS row stride of the candidate tile
constexpr int kKnnMaxK = 32;          // neighbours, at most
constexpr int kKnnParts = 16;         // parts of the candidates, at most
constexpr int kKnnSlots = 512;        // workgroups on the chip at a time (two per CU)

struct KnnArgs {
  const float* P;  // tiles of (4 SM + 1) x 64: dimensions, then norms
  int n, k, parts, tiles, tiles_per_part, root;
  unsigned long long* part;  // n x parts x k keys (parts > 1)
  int* idx;                  // n x k neighbour indices, nearest first
  float* dist;               // n x k distances
};

typedef unsigned long long knn_key;  // distance in the high word, index in the low one

__device__ __forceinline__ knn_key knn_make_key(float v, int id) {
  const int b = __builtin_bit_cast(int, v);
  const unsigned m = (unsigned)b ^ (unsigned)((b >> 31) | (int)0x80000000);  // order-preserving
  return ((knn_key)m << 32) | (unsigned)id;
}
__device__ __forceinline__ float knn_key_dist(knn_key key) {
  const unsigned m = (unsigned)(key >> 32);
  return __builtin_bit_cast(float, (m & 0x80000000u) ? m ^ 0x80000000u : ~m);
}

// Tiles of 64 rows: dimension c of row 64 t + i at P[t][c][i]; rows past n and
// dimensions past d are zero.  The last line holds the squared row norm (sum
// in FP64, rounded once), for cosine 1, and infinity past n; cosine rows are
// scaled to unit length.  One workgroup per tile.
static __global__ __launch_bounds__(kBlock) void knn_pack_kernel(const float* __restrict__ X,
                                                                 float* __restrict__ P,
                                                                 long long n, int d, int dp,
                                                                 int cosine) {
  extern __shared__ __align__(16) float pack_smem[];  // (dp + 1) x 65
  constexpr int PS = kKnnC + 1;
  const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
  const long long row0 = (long long)blockIdx.x * kKnnC;
  for (int i = wv; i < kKnnC; i += kBlock / kWave) {
    const long long r = row0 + i;
    float v[2];
    double s = 0.0;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int c = lane + u * kWave;
      v[u] = (r < n && c < d) ? X[r * d + c] : 0.f;
      s += (double)v[u] * (double)v[u];
    }
    s = wave_sum(s);
    const double inv = s > 0.0 ? 1.0 / sqrt(s) : 0.0;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int c = lane + u * kWave;
      if (c < dp) pack_smem[c * PS + i] = (cosine && c < d) ? (float)(v[u] * inv) : v[u];
    }
    if (lane == 0) pack_smem[dp * PS + i] = r >= n ? INFINITY : cosine ? 1.f : (float)s;
  }
  __syncthreads();
  float* out = P + (long long)blockIdx.x * (dp + 1) * kKnnC;
  for (int e = threadIdx.x; e < (dp + 1) * kKnnC; e += kBlock)
    out[e] = pack_smem[(e / kKnnC) * PS + e % kKnnC];
}

// Entries per query buffer: the k kept ones, and 16 more than the largest
// count at which the next 16 candidates are still appended without a cut.
// 48 and 60 leave room for two workgroups per CU up to 52 (k > 16) and 100
// dimensions (k <= 16).
__host__ __device__ constexpr int knn_cap(int KM) { return KM <= 16 ? 48 : 60; }

template <int SM, int KM>
constexpr size_t knn_lds() {
  return (size_t)(4 * SM + 1) * kKnnCS * sizeof(float) +
         (size_t)kKnnQ * knn_cap(KM) * (sizeof(float) + sizeof(int));
}

// What bounds it: the FP32 matrix cores (4 SM instructions of 32 cycles per
// wave and tile; 60k rows x 50 without any append: 3.3 ms, 2.4 at the rate of a
// large matrix product), then appends and cuts, which are dense for the first
// few thousand candidates (4.1 ms with them).  Sixteen queries a wave leave
// registers and LDS for four waves per SIMD, whose products run while others
// test, append or wait: 20k rows x 50, k = 15: 0.70 ms (4.7 ms with sorted
// lists in registers, which every lane of a wave walked for each insertion;
// 0.95 ms with 32 queries a wave); 150k x 30, k = 30, cosine: 18.9 ms (193).
template <int SM, int KM, bool COS>
__global__ __launch_bounds__(kKnnThreads, 4) void knn_kernel(KnnArgs a) {
  constexpr int D1 = 4 * SM + 1, CAP = knn_cap(KM), LIM = CAP - 16;
  constexpr int NF4 = (D1 * (kKnnC / 4) + kKnnThreads - 1) / kKnnThreads;  // 16-byte loads per thread
  static_assert(LIM >= KM && CAP <= kWave && CAP % 4 == 0, "query buffer");
  extern __shared__ __align__(16) float knn_smem[];
  float(*s_ct)[kKnnCS] = reinterpret_cast<float(*)[kKnnCS]>(knn_smem);
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int lr = lane & 15, lg = lane >> 4;
  float* s_bd = knn_smem + D1 * kKnnCS + wv * 16 * CAP;  // buffers: distances, indices
  int* s_bi = reinterpret_cast<int*>(knn_smem + D1 * kKnnCS + kKnnQ * CAP) + wv * 16 * CAP;
  const int n = a.n, k = a.k;
  const int group = blockIdx.x / a.parts, part = blockIdx.x - group * a.parts;
  const int q0 = group * kKnnQ + wv * 16;
  const int t0 = part * a.tiles_per_part, t1 = min(a.tiles, t0 + a.tiles_per_part);

  // A operand (queries q0 + lr, dimensions 4 s + lg), held for the whole
  // stream; the norm, threshold and count of the D-fragment rows this lane
  // holds (4 lg + r).  A query past n passes nothing.
  float za[SM], qn[4], thr[4];
  int cnt[4];
  {
    const float* src = a.P + (long long)min(q0 / kKnnC, a.tiles - 1) * D1 * kKnnC + q0 % kKnnC;
#pragma unroll
    for (int s = 0; s < SM; ++s) za[s] = src[(4 * s + lg) * kKnnC + lr];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      qn[r] = src[4 * SM * kKnnC + 4 * lg + r];
      thr[r] = (q0 + 4 * lg + r < n) ? INFINITY : -INFINITY;
      cnt[r] = 0;
    }
  }

  // the loads above end here: a wait for them inside the loop would be one for
  // the tile in flight too
#pragma unroll
  for (int s = 0; s < SM; ++s) asm volatile("" : "+v"(za[s]));
#pragma unroll
  for (int r = 0; r < 4; ++r) asm volatile("" : "+v"(qn[r]));

  // The k nearest of four queries at once, each sorted to the front of its
  // buffer: the 16 lanes of group lg hold the c entries of row 4 lg + r.  An
  // entry's place is the number of smaller distances and, among equal ones
  // (which the read-back of the places detects), of earlier entries: entries
  // of one distance stand in index order.  Returns the row's k-th distance
  // (infinity while there are fewer than k).
  auto cut = [&](int r, int c) __attribute__((always_inline)) -> float {
    constexpr int E = (CAP + 15) / 16;
    float* bd = s_bd + (4 * lg + r) * CAP;
    int* bi = s_bi + (4 * lg + r) * CAP;
    float v[E];
    int id[E], rank[E];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int at = lr + 16 * e;
      v[e] = (at < c) ? bd[at] : INFINITY;
      id[e] = (at < c) ? bi[at] : -1;
      rank[e] = 0;
      if (at >= c && at < CAP) bd[at] = INFINITY;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll 4
    for (int i = 0; i < CAP; i += 4) {
      const floatx4 o = *reinterpret_cast<const floatx4*>(bd + i);
#pragma unroll
      for (int e = 0; e < E; ++e)
        rank[e] += (int)(o.x < v[e]) + (int)(o.y < v[e]) + (int)(o.z < v[e]) + (int)(o.w < v[e]);
    }
    auto put = [&]() __attribute__((always_inline)) {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
      for (int e = 0; e < E; ++e)
        if (lr + 16 * e < c && rank[e] < k) bi[rank[e]] = id[e];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    };
    put();
    bool lost = false;
#pragma unroll
    for (int e = 0; e < E; ++e)
      if (lr + 16 * e < c && rank[e] < k) lost |= bi[rank[e]] != id[e];
    if (__builtin_amdgcn_ballot_w64(lost)) {
#pragma unroll 1
      for (int i = 0; i < CAP; ++i) {
        const float o = bd[i];
#pragma unroll
        for (int e = 0; e < E; ++e) rank[e] += (int)(o == v[e] && i < lr + 16 * e);
      }
      put();
    }
#pragma unroll
    for (int e = 0; e < E; ++e)
      if (lr + 16 * e < c && rank[e] < k) bd[rank[e]] = v[e];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    return (c >= k) ? bd[k - 1] : INFINITY;
  };

  floatx4 pre[NF4];  // the next tile, on its way from L2
  auto load_tile = [&](int t) __attribute__((always_inline)) {
    const floatx4* src = reinterpret_cast<const floatx4*>(a.P + (long long)t * D1 * kKnnC);
#pragma unroll
    for (int u = 0; u < NF4; ++u) pre[u] = src[min(tid + u * kKnnThreads, D1 * (kKnnC / 4) - 1)];
  };
  if (t0 < t1) load_tile(t0);
  for (int t = t0; t < t1; ++t) {
    __syncthreads();
#pragma unroll
    for (int u = 0; u < NF4; ++u) {
      const int e = tid + u * kKnnThreads;
      if (e < D1 * (kKnnC / 4))
        *reinterpret_cast<floatx4*>(&s_ct[e / (kKnnC / 4)][4 * (e % (kKnnC / 4))]) = pre[u];
    }
    __syncthreads();
    if (t + 1 < t1) load_tile(t + 1);
    floatx4 acc[4];
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) acc[ct] = floatx4{0.f, 0.f, 0.f, 0.f};
    // the next step's operand is read while this one's products run
    float b[2][4];
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) b[0][ct] = s_ct[lg][16 * ct + lr];
#pragma unroll
    for (int s = 0; s < SM; ++s) {
      if (s + 1 < SM) {
#pragma unroll
        for (int ct = 0; ct < 4; ++ct) b[(s + 1) & 1][ct] = s_ct[4 * (s + 1) + lg][16 * ct + lr];
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ct = 0; ct < 4; ++ct) acc[ct] = mfma_f32(za[s], b[s & 1][ct], acc[ct]);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) {
      const int id = t * kKnnC + 16 * ct + lr;
      const float cn = s_ct[4 * SM][16 * ct + lr];
      float dd[4];
      unsigned long long pass[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float dot = acc[ct][r];
        dd[r] = COS ? 1.f - dot : fmaxf(qn[r] + cn - 2.f * dot, 0.f);
        // a later candidate at the threshold itself has the higher index
        pass[r] = __builtin_amdgcn_ballot_w64(dd[r] < thr[r]);
      }
      if ((pass[0] | pass[1] | pass[2] | pass[3]) == 0) continue;
      const unsigned long long real = __builtin_amdgcn_ballot_w64(id < n);
      unsigned long long full = 0;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        // the 16 lanes of a row append in index order
        const unsigned long long m = pass[r] & real;
        if (m == 0) continue;
        const unsigned half = lg < 2 ? (unsigned)m : (unsigned)(m >> 32);
        const unsigned bits = __builtin_amdgcn_ubfe(half, 16 * (lg & 1), 16);
        if (dd[r] < thr[r] && id < n) {
          const int at = (4 * lg + r) * CAP + cnt[r] + __builtin_popcount(bits & ((1u << lr) - 1u));
          s_bd[at] = dd[r];
          s_bi[at] = id;
        }
        cnt[r] += __builtin_popcount(bits);
        full |= __builtin_amdgcn_ballot_w64(cnt[r] > LIM);
      }
      if (full) {
#pragma unroll 1
        for (int r = 0; r < 4; ++r) {
          const int c = r == 0 ? cnt[0] : r == 1 ? cnt[1] : r == 2 ? cnt[2] : cnt[3];
          if (__builtin_amdgcn_ballot_w64(c > LIM) == 0) continue;
          const float kth = cut(r, c);
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            cnt[u] = (u == r) ? min(c, k) : cnt[u];
            thr[u] = (u == r) ? fminf(thr[u], kth) : thr[u];
          }
        }
      }
    }
  }

  // sorted lists of this part; a query with fewer than k candidates ends in
  // (FLT_MAX, -1)
#pragma unroll 1
  for (int r = 0; r < 4; ++r) {
    const int c = r == 0 ? cnt[0] : r == 1 ? cnt[1] : r == 2 ? cnt[2] : cnt[3];
    cut(r, c);
    const int row = 4 * lg + r;
    const long long q = q0 + row;
    if (q >= n) continue;
    for (int e = lr; e < k; e += 16) {
      const float v = (e < c) ? s_bd[row * CAP + e] : FLT_MAX;
      const int id = (e < c) ? s_bi[row * CAP + e] : -1;
      if (a.parts > 1) {
        a.part[(q * a.parts + part) * k + e] = knn_make_key(v, id);
      } else {
        a.idx[q * k + e] = id;
        a.dist[q * k + e] = a.root ? sqrtf(v) : v;
      }
    }
  }
}

// The k nearest of a query from its parts' sorted lists (one wave per query):
// an entry's place is its own position plus, by bisection, the number of
// smaller keys in every other list (equal keys, which are (FLT_MAX, -1) only,
// go by list).
static __global__ __launch_bounds__(kBlock) void knn_merge_kernel(KnnArgs a) {
  __shared__ knn_key s_l[kBlock / kWave][kKnnParts * kKnnMaxK];
  const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
  const long long q = (long long)blockIdx.x * (kBlock / kWave) + wv;
  const int k = a.k, tot = a.parts * k;
  if (q < a.n)
    for (int e = lane; e < tot; e += kWave) s_l[wv][e] = a.part[q * tot + e];
  __syncthreads();
  if (q >= a.n) return;
  const knn_key* L = s_l[wv];
  for (int e = lane; e < tot; e += kWave) {
    const int l = e / k;
    const knn_key key = L[e];
    int place = e - l * k;
    for (int o = 0; o < a.parts && place < k; ++o) {
      if (o == l) continue;
      int lo = 0, hi = k;
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        const knn_key v = L[o * k + mid];
        if (v < key || (v == key && o < l))
          lo = mid + 1;
        else
          hi = mid;
      }
      place += lo;
    }
    if (place < k) {
      const float v = knn_key_dist(key);
      a.idx[q * k + place] = (int)(unsigned)key;
      a.dist[q * k + place] = a.root ? sqrtf(v) : v;
    }
  }
}

// UMAP fuzzy-set membership of every kNN edge, one thread per row: the
// smooth-kNN distance normalisation of umap-learn's smooth_knn_dist
// (local_connectivity = 1, bandwidth = 1: rho = the nearest non-zero
// distance; sigma from 64 bisection steps on
// sum_{j >= 1} exp(-max(0, d_j - rho) / sigma) = log2(k), tolerance 1e-5,
// floored at 1e-3 times the row's mean distance (the global mean when
// rho = 0)), then compute_membership_strengths: w = 0 for the row itself,
// 1 when d <= rho or sigma = 0, exp(-(d - rho) / sigma) otherwise.  The
// reference gets the same quantities from cuML's fuzzy_simplicial_set
// (preprocessing/_neighbors/_neighbors.py:134-159).
static __global__ void umap_membership_kernel(const float* __restrict__ dist,
                                              const int* __restrict__ idx, long long n, int k,
                                              double mean_all, float* __restrict__ w,
                                              float* __restrict__ sigmas, float* __restrict__ rhos) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float* di = dist + i * k;
  double rho = 0.0, mean_i = 0.0;
  bool have = false;
  for (int j = 0; j < k; ++j) {
    const double v = di[j];
    mean_i += v;
    if (!have && v > 0.0) {
      rho = v;
      have = true;
    }
  }
  mean_i /= k;
  const double target = log2((double)k);
  double lo = 0.0, hi = INFINITY, mid = 1.0;
  for (int it = 0; it < 64; ++it) {
    double psum = 0.0;
    for (int j = 1; j < k; ++j) {
      const double dd = (double)di[j] - rho;
      psum += dd > 0.0 ? exp(-(dd / mid)) : 1.0;
    }
    if (fabs(psum - target) < 1e-5) break;
    if (psum > target) {
      hi = mid;
      mid = (lo + hi) / 2.0;
    } else {
      lo = mid;
      mid = isinf(hi) ? mid * 2.0 : (lo + hi) / 2.0;
    }
  }
  double sigma = mid;
  const double floor_v = 1e-3 * (rho > 0.0 ? mean_i : mean_all);
  if (sigma < floor_v) sigma = floor_v;
  for (int j = 0; j < k; ++j) {
    const double dd = (double)di[j] - rho;
    double v;
    if (idx[i * k + j] == (int)i)
      v = 0.0;
    else if (dd <= 0.0 || sigma == 0.0)
      v = 1.0;
    else
      v = exp(-(dd / sigma));
    w[i * k + j] = (float)v;
  }
  if (sigmas) sigmas[i] = (float)sigma;
  if (rhos) rhos[i] = (float)rho;
}

static int knn_sm(int d) {
  const int s = (d + 3) / 4;
  return s <= 4 ? 4 : s <= 8 ? 8 : s <= 13 ? 13 : s <= 16 ? 16 : s <= 25 ? 25 : s <= 32 ? 32 : 0;
}

template <int SM, int KM, bool COS>
static int launch_knn_one(const KnnArgs& a, int grid, hipStream_t s) {
  constexpr size_t lds = knn_lds<SM, KM>();
  HZ_TRY(prepare_lds(reinterpret_cast<const void*>(knn_kernel<SM, KM, COS>), lds));
  hipLaunchKernelGGL((knn_kernel<SM, KM, COS>), dim3(grid), dim3(kKnnThreads), lds, s, a);
  return HZ_OK;
}

template <int SM>
static int launch_knn_sm(const KnnArgs& a, bool cosine, int grid, hipStream_t s) {
  if (a.k <= 16)
    return cosine ? launch_knn_one<SM, 16, true>(a, grid, s)
                  : launch_knn_one<SM, 16, false>(a, grid, s);
  return cosine ? launch_knn_one<SM, 32, true>(a, grid, s)
                : launch_knn_one<SM, 32, false>(a, grid, s);
}

// Parts the candidates are split into: the number with the shortest time, in
// candidates streamed by a workgroup that has its CU to itself.  Two that share
// a CU take 1.47 times as long each, and every part pays again, like
// kKnnSettle more candidates, until its thresholds have settled.  Measured at
// 20k rows x 50 (157 groups of queries): 1.07 ms in one part, 0.70 in three
// (471 workgroups), 0.90 in four; 5k: 0.39 ms in one, 0.144 in six; 60k
// (469 groups): 4.1 ms in one, 4.4 in two; 150k x 30, k = 30: 18.9 and 20.6.
// Above 52 dimensions with k > 16 the LDS holds one workgroup per CU, not two; the
// rule is the same there: 10k x 100, k = 30 0.64 ms in the three it picks, 0.64 at
// best; 80k 17.2 and 17.2; 40k 7.0 in one, 6.0 in three.
constexpr long long kKnnSettle = 15000;
// The parts' lists stay within 128 MiB: past that a second part saves 2% at most
// where it saves anything (664k x 50, k = 15: 399 ms, 401 in one part; k = 30:
// 270k x 50 79.8 and 79.1, 400k x 30 118.3 and 113.7).
constexpr long long kKnnListBytes = 128LL << 20;
static int knn_parts(long long n, int k) {
  const long long groups = ceil_div(n, kKnnQ);
  int best = 1;
  long long best_cost = 0;
  for (int p = 1; p <= std::min<long long>(kKnnParts, ceil_div(n, kKnnC)); ++p) {
    if (p > 1 && n * p * k * (long long)sizeof(knn_key) > kKnnListBytes) break;
    const long long full = groups * p / kKnnSlots, rest = groups * p % kKnnSlots;
    const long long rounds = 147 * full + (rest == 0 ? 0 : rest <= kKnnSlots / 2 ? 100 : 147);
    const long long cost = rounds * (ceil_div(n, p) + kKnnSettle);
    if (p == 1 || cost < best_cost) {
      best = p;
      best_cost = cost;
    }
  }
  return best;
}

struct KnnLayout {
  int sm, tiles, parts;
  float* P;
  knn_key* part;
  size_t bytes;
};

static void knn_layout(long long n, int d, int k, void* base, KnnLayout& L) {
  L.sm = knn_sm(d);
  L.tiles = (int)ceil_div(n, kKnnC);
  L.parts = knn_parts(n, k);
  Carve c(base);
  L.P = c.take<float>((size_t)L.tiles * (4 * L.sm + 1) * kKnnC);
  L.part = c.take<knn_key>(L.parts > 1 ? (size_t)n * L.parts * k : 0);
  L.bytes = align_up(c.off, 256);
}

}  // namespace hz

using namespace hz;

extern "C" {

size_t hz_knn_workspace_bytes_k(long long n_rows, int n_cols, int metric, int k) {
  (void)metric;
  if (n_rows < 1 || n_cols < 1 || k < 1 || k > kKnnMaxK) return 0;
  KnnLayout L;
  knn_layout(n_rows, n_cols, k, nullptr, L);
  return L.bytes;
}

size_t hz_knn_workspace_bytes(long long n_rows, int n_cols, int metric) {
  size_t most = 0;
  for (int k = 1; k <= kKnnMaxK; ++k)
    most = std::max(most, hz_knn_workspace_bytes_k(n_rows, n_cols, metric, k));
  return most;
}

int hz_knn(int metric, const float* X, long long n_rows, int n_cols, int k, int32_t* indices,
           float* distances, void* ws, size_t ws_bytes, void* stream) {
  HZ_RET_IF(metric != HZ_KNN_EUCLIDEAN && metric != HZ_KNN_SQEUCLIDEAN && metric != HZ_KNN_COSINE,
            HZ_ERR_ARG, "unknown metric %d", metric);
  HZ_RET_IF(n_rows < 1 || n_cols < 1 || k < 1, HZ_ERR_ARG, "bad shape (n=%lld d=%d k=%d)", n_rows,
            n_cols, k);
  HZ_RET_IF(k > n_rows, HZ_ERR_ARG, "k=%d exceeds the %lld rows", k, n_rows);
  HZ_RET_IF(k > kKnnMaxK, HZ_ERR_UNSUPPORTED, "k=%d > %d neighbours is not supported", k, kKnnMaxK);
  HZ_RET_IF(n_rows >= (1LL << 31) - kKnnQ, HZ_ERR_UNSUPPORTED, "too many rows");
  const int sm = knn_sm(n_cols);
  HZ_RET_IF(sm == 0, HZ_ERR_UNSUPPORTED, "n_cols=%d > 128 is not supported", n_cols);
  HZ_RET_IF(!X || !indices || !distances, HZ_ERR_ARG, "X, indices and distances are required");
  const size_t need = hz_knn_workspace_bytes_k(n_rows, n_cols, metric, k);
  HZ_RET_IF(!ws || ws_bytes < need, HZ_ERR_WORKSPACE, "workspace too small: %zu < %zu", ws_bytes,
            need);
  hipStream_t s = static_cast<hipStream_t>(stream);
  KnnLayout L;
  knn_layout(n_rows, n_cols, k, ws, L);
  const bool cosine = metric == HZ_KNN_COSINE;
  hipLaunchKernelGGL(knn_pack_kernel, dim3(L.tiles), dim3(kBlock),
                     (4 * sm + 1) * (kKnnC + 1) * sizeof(float), s, X, L.P, n_rows, n_cols, 4 * sm,
                     (int)cosine);
  HZ_LAUNCHED("knn_pack_kernel");
  KnnArgs a;
  a.P = L.P;
  a.n = (int)n_rows;
  a.k = k;
  a.tiles = L.tiles;
  a.tiles_per_part = (int)ceil_div(L.tiles, L.parts);
  a.parts = (int)ceil_div(L.tiles, a.tiles_per_part);
  a.root = metric == HZ_KNN_EUCLIDEAN;
  a.part = L.part;
  a.idx = indices;
  a.dist = distances;
  const int grid = (int)ceil_div(n_rows, kKnnQ) * a.parts;
  switch (sm) {
    case 4: HZ_TRY(launch_knn_sm<4>(a, cosine, grid, s)); break;
    case 8: HZ_TRY(launch_knn_sm<8>(a, cosine, grid, s)); break;
    case 13: HZ_TRY(launch_knn_sm<13>(a, cosine, grid, s)); break;
    case 16: HZ_TRY(launch_knn_sm<16>(a, cosine, grid, s)); break;
    case 25: HZ_TRY(launch_knn_sm<25>(a, cosine, grid, s)); break;
    default: HZ_TRY(launch_knn_sm<32>(a, cosine, grid, s)); break;
  }
  HZ_LAUNCHED("knn_kernel");
  if (a.parts > 1) {
    hipLaunchKernelGGL(knn_merge_kernel, dim3((int)ceil_div(n_rows, kBlock / kWave)), dim3(kBlock), 0,
                       s, a);
    HZ_LAUNCHED("knn_merge_kernel");
  }
  return HZ_OK;
}

int hz_umap_weights(const float* distances, const int32_t* indices, long long n_rows, int k,
                    double mean_distance, float* weights, float* sigmas, float* rhos,
                    void* stream) {
  HZ_RET_IF(n_rows < 1 || k < 2, HZ_ERR_ARG, "bad shape (n=%lld k=%d)", n_rows, k);
  HZ_RET_IF(!distances || !indices || !weights, HZ_ERR_ARG,
            "distances, indices and weights are required");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int grid = (int)((n_rows + 255) / 256);
  hipLaunchKernelGGL(umap_membership_kernel, dim3(grid), dim3(256), 0, s, distances, indices,
                     n_rows, k, mean_distance, weights, sigmas, rhos);
  HZ_LAUNCHED("umap_membership_kernel");
  return HZ_OK;
}

}  // extern "C"
