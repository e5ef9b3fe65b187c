// Block sweep of FP64 jobs: all blocks of one clustering iteration in one
// cooperative launch (the block loop of clustering.cu:308-372; the protocol
// between workgroups is that of hz_sweep.hpp: every workgroup keeps the same
// O and E, the new rows' sums are exchanged through counted accumulators).
//
// What differs from the FP32 sweep:
//  * 512 threads: two waves per SIMD, so one wave's FP64 exponentials run
//    beside the other's v_mfma_f64_16x16x4 chain (64 cycles per instruction).
//  * O and E live in the workgroup's own device memory, read by the threads
//    that read the block sums (one cluster column, every GB-th batch each), which
//    leaves the LDS to the centroids: 100 PCs x 100 clusters x 32 batches still
//    fit.
//  * A wait that runs out leaves O, E and the history as they were, so that the
//    caller can do the iteration again with one launch per block.
//  * A block sum is exchanged in two words of the fixed-point value (31 low
//    bits, then the rest), each with its own contribution count above bit 53,
//    so the sums keep 61 bits: the scale is 2^min(52, 61 - bitlen(bs + 1)),
//    finer than the per-block path's by the ratio of cells to block size.
//  * exp(term (1 - sim)) pen is one exponential, of term (1 - sim) + log pen;
//    the entropy's logarithm is that argument minus the row sum's logarithm,
//    plus the part that the reference's log(x + 1e-12) adds (log1p_eps).
// What bounds it: at 1.3M cells (d = 50, K = 100, 16 batches) FP64 work (the
// MFMA chain and 130M exponentials per iteration): 726 us per clustering
// iteration, 36 us a block (106 us a row launch with one launch per block); the
// matrix pipes are busy 29% of the time, the waves (two per SIMD) wait 29% of
// theirs.  Below about 100k cells the chain of block exchanges: 2.7k cells 13 us
// a block against 36 us, 37k cells x 100 PCs x 32 batches 19 against 51.
#pragma once

#include "hz_sweep.hpp"

namespace hz {

typedef double doublex2 __attribute__((ext_vector_type(2)));
typedef double doublex4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

// D[4 r + l / 16][l % 16] of lane l, register r; A[l % 16][l / 16] and
// B[l / 16][l % 16] as the FP32 shape (checked on gfx950).
__device__ __forceinline__ doublex4 mfma_f64(double a, double b, doublex4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

constexpr int kSw64Threads = 512;
constexpr int kSw64Waves = kSw64Threads / kWave;
constexpr int kSw64Rounds = 8;    // rounds of a block whose chunks are staged one block ahead
constexpr int kSw64Entry = 3 + kChunkRows;  // ints per staged chunk: seg, len, start, cells
constexpr int kSw64U = 8;         // batches per update thread, at most
constexpr int kSplitBits = 31;    // low word of a block sum
constexpr int kSw64GaveUp = 1 << 24;  // in the count of final arrivals: a wait ran out

struct Sweep64Args {
  const double* Z;
  const double* YT;  // d x Kp
  double* R;
  const int* order;
  const int* seg_ch;
  const int* ch_start;
  const int* ch_len;
  const int* ch_seg;
  const long long* acc_in;   // nseg x K, old-row sums (complete at launch)
  long long* acc_out;        // low words, then high words rep_stride apart; zero at launch
  long long* obj_acc;        // kRep x 2, zero at launch
  const int* cnt;            // nblk x B contributions per block sum
  long long rep_stride;
  double* O;
  double* E;
  const double* Pr;
  const double* theta;
  Ctrl* ctrl;
  double* last_obj;
  int n, d, K, Kp, B, nblk;
  double term, sigma, tol;
  int stabilized;
  double inv_scale_o, scale_obj, inv_scale_obj;
  double* oe;  // 2 x B x K per workgroup: its copy of O and E
  double scale_blk, inv_scale_blk;  // scale of the block sums (acc_out)
  unsigned spin_limit;
};

// LDS row stride (doubles) of the staged centroids, 16 mod 32: two lane groups
// of a fragment read cover the 64 banks.
__host__ __device__ constexpr int sw64_stride(int NT) {
  return 16 * NT % 32 == 16 ? 16 * NT : 16 * NT + 16;
}

__host__ __device__ inline size_t sweep64_lds(int SM, int NT, int B, int K, int nblk) {
  return (size_t)4 * SM * sw64_stride(NT) * 8 + (size_t)2 * B * K * 8 +
         (size_t)2 * kSw64Threads * 8 + (size_t)2 * B * 8 +
         (size_t)2 * kSw64Rounds * kSw64Waves * kSw64Entry * 4 + (size_t)nblk * 4 * 4;
}

// Column that lane group lg supplies to k-step s: two k-steps share a 16-byte
// load whose four lane groups read 64 contiguous bytes of a row; the last of
// an odd number of k-steps takes four adjacent columns.
template <int SM>
__device__ __forceinline__ constexpr int z64_col(int s, int lg) {
  return s < (SM & ~1) ? 8 * (s >> 1) + 2 * lg + (s & 1) : 4 * s + lg;
}

// x log(x + 1e-12) - x log x = x log1p(1e-12 / x) for x >= 0.  At most 1e-12,
// so FP32 holds it to 1e-18.
__device__ __forceinline__ float log1p_eps(float x) {
  x = fmaxf(x, 1e-30f);
  const float u = 1e-12f * __builtin_amdgcn_rcpf(x);
  const float l = u < 1e-3f ? u * (1.f - 0.5f * u)
                            : 0.693147180559945309f * __builtin_amdgcn_logf(1.f + u);
  return x * l;
}

// Sum over each group of 16 lanes (the DPP steps of the FP32 sum16, on both
// halves of the value).
__device__ __forceinline__ double sum16(double v) {
  auto step = [](double x, auto ctrl) __attribute__((always_inline)) {
    const u32x2 b = __builtin_bit_cast(u32x2, x);
    u32x2 o;
    o.x = (unsigned)__builtin_amdgcn_update_dpp(0, (int)b.x, decltype(ctrl)::value, 0xF, 0xF, false);
    o.y = (unsigned)__builtin_amdgcn_update_dpp(0, (int)b.y, decltype(ctrl)::value, 0xF, 0xF, false);
    return x + __builtin_bit_cast(double, o);
  };
  v = step(v, std::integral_constant<int, 0xB1>{});
  v = step(v, std::integral_constant<int, 0x4E>{});
  v = step(v, std::integral_constant<int, 0x141>{});
  return step(v, std::integral_constant<int, 0x140>{});
}

// exp(x) = 2^n exp(r), n = round(x / ln 2), |r| <= ln 2 / 2: two-part ln 2,
// Taylor series to r^13 / 13! (the next term is below 5e-18).  Where the result
// is not zero, |n| <= 1075 and the two parts' remainder is below 1e-22; further
// down the result is zero as long as n fits an int: x > -1.4e9, which the padded
// columns' -1e5 - 2 / sigma stays above for sigma > 2e-9.
__device__ __forceinline__ double exp64(double x) {
  const double n = __builtin_rint(x * 0x1.71547652b82fep+0);
  double r = fma(n, -0x1.62e42feep-1, x);
  r = fma(n, -0x1.a39ef35793c76p-33, r);
  double p = 1.0 / 6227020800.0;
  p = fma(p, r, 1.0 / 479001600.0);
  p = fma(p, r, 1.0 / 39916800.0);
  p = fma(p, r, 1.0 / 3628800.0);
  p = fma(p, r, 1.0 / 362880.0);
  p = fma(p, r, 1.0 / 40320.0);
  p = fma(p, r, 1.0 / 5040.0);
  p = fma(p, r, 1.0 / 720.0);
  p = fma(p, r, 1.0 / 120.0);
  p = fma(p, r, 1.0 / 24.0);
  p = fma(p, r, 1.0 / 6.0);
  p = fma(p, r, 0.5);
  p = fma(p, r, 1.0);
  p = fma(p, r, 1.0);
  return __builtin_amdgcn_ldexp(p, (int)n);
}

// Keeps a running sum where it stands in the code: the optimiser otherwise
// moves the adds to the sum's use and keeps every term in registers till then.
template <typename T>
__device__ __forceinline__ void pin(T& x) {
  asm volatile("" : "+v"(x));
}

// The same value, but not known to the optimiser to be unchanged: what is
// derived from it is computed where it is used instead of being kept (and
// spilled) across the block loop.
__device__ __forceinline__ int fresh(int x) {
  asm volatile("" : "+v"(x));
  return x;
}
__device__ __forceinline__ int fresh_s(int x) {
  asm volatile("" : "+s"(x));
  return x;
}

template <int NT, int SM>
__global__ __launch_bounds__(kSw64Threads) void sweep64_kernel(Sweep64Args a) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int NW = kSw64Waves, NTH = kSw64Threads;
  constexpr int YS = sw64_stride(NT);
  __shared__ int s_last;
  __shared__ double red[NW];
  __shared__ double s_obj[NW][2];
  Ctrl* ctrl = a.ctrl;
  // the same in every workgroup, unless a wait of this launch ran out already
  if (ctrl->done || ctrl->pad0) return;
  const int wg = blockIdx.x, G = gridDim.x;
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int lr = lane & 15, lg = lane >> 4;
  const int d = a.d, K = a.K, B = a.B, BK = B * K;

  double* Ys = reinterpret_cast<double*>(smem);                  // 4 SM x YS
  double* s_lpen = Ys + 4 * SM * YS;                             // B x K: log penalty
  unsigned long long* s_dO = reinterpret_cast<unsigned long long*>(s_lpen + BK);  // B x K
  double* s_co = reinterpret_cast<double*>(s_dO + BK);           // column partials: new rows
  double* s_ci = s_co + NTH;                                     // column partials: old rows
  double* s_pr = s_ci + NTH;
  double* s_th = s_pr + B;
  int* s_tab = reinterpret_cast<int*>(s_th + B);  // 2 x rounds x waves x entry
  int* s_lohi = s_tab + 2 * kSw64Rounds * NW * kSw64Entry;  // nblk x 4: chunks, batches

  // chunk range and batch range of this workgroup in every block
  for (int j = tid; j < a.nblk; j += NTH) {
    const int nlo = a.seg_ch[j * B], nhi = a.seg_ch[j * B + B];
    const int per = (nhi - nlo + G - 1) / G;
    const int lo = nlo + wg * per;
    const int hi = min(nhi, lo + per);
    s_lohi[4 * j] = lo;
    s_lohi[4 * j + 1] = hi;
    s_lohi[4 * j + 2] = (lo < hi) ? a.ch_seg[lo] - j * B : 0;
    s_lohi[4 * j + 3] = (lo < hi) ? a.ch_seg[hi - 1] - j * B : -1;
  }
  for (int b = tid; b < B; b += NTH) {
    s_pr[b] = a.Pr[b];
    s_th[b] = a.theta[b];
  }
  // normalised centroids; rows past d and columns past K are zero
  for (int e0 = tid; e0 < 4 * SM * 16 * NT; e0 += 8 * NTH) {
    double y[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int e = e0 + u * NTH;
      const int c = e / (16 * NT), k = e % (16 * NT);
      y[u] = a.YT[(long long)min(c, d - 1) * a.Kp + min(k, K - 1)];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int e = e0 + u * NTH;
      const int c = e / (16 * NT), k = e % (16 * NT);
      if (c < 4 * SM) Ys[c * YS + k] = (c < d && k < K) ? y[u] : 0.0;
    }
  }

  // this thread's part of the workgroup's O and E: cluster ck, batches cg,
  // cg + GB, ...  It stays in the thread's own memory (L2), read while the
  // block sums are polled: neither registers nor LDS hold it during the rows.
  const int GB = NTH / K;
  const int ck = tid % K, cg = tid / K;
  const bool upd = tid < GB * K;
  double* my_o = a.oe + (size_t)wg * 2 * BK + ck;
#pragma unroll
  for (int u = 0; u < kSw64U; ++u) {
    const int b = cg + u * GB;
    if (upd && b < B) {
      my_o[b * K] = a.O[b * K + ck];
      my_o[BK + b * K] = a.E[b * K + ck];
    }
  }
  __syncthreads();

  // chunks of rounds 0 .. kSw64Rounds - 1 of block j, for every wave: entry
  // (round, wave) of buffer j % 2.  Descriptors, then cell ids (two steps with
  // a barrier after each, so that the caller can put work between them).
  auto entry = [&](int j, int r, int w) __attribute__((always_inline)) {
    return s_tab + (((j & 1) * kSw64Rounds + r) * NW + w) * kSw64Entry;
  };
  int ds = -1, dl = 0, dp = 0;  // thread (round, wave): segment, length, start
  auto load_desc = [&](int j) __attribute__((always_inline)) {
    if (tid < kSw64Rounds * NW) {
      const int c = s_lohi[4 * j] + tid;
      const bool has = c < s_lohi[4 * j + 1];
      ds = has ? a.ch_seg[c] : -1;
      dl = has ? a.ch_len[c] : 0;
      dp = has ? a.ch_start[c] : 0;
    }
  };
  auto put_desc = [&](int j) __attribute__((always_inline)) {
    if (tid < kSw64Rounds * NW) {
      int* e = entry(j, tid / NW, tid % NW);
      e[0] = ds;
      e[1] = dl;
      e[2] = dp;
    }
  };
  constexpr int kCellU = kSw64Rounds * NW * kChunkRows / NTH;
  auto load_cells = [&](int j, int (&x)[kCellU]) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kCellU; ++u) {
      const int q = tid + u * NTH, row = q % kChunkRows;
      const int* e = entry(j, q / (NW * kChunkRows), q / kChunkRows % NW);
      x[u] = a.order[(row < e[1]) ? e[2] + row : 0];  // order[0] is always valid
    }
  };
  auto put_cells = [&](int j, const int (&x)[kCellU]) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kCellU; ++u) {
      const int q = tid + u * NTH;
      entry(j, q / (NW * kChunkRows), q / kChunkRows % NW)[3 + q % kChunkRows] = x[u];
    }
  };

  struct Chunk {
    int seg, len, cell;  // cell: of row `lane` (lane < 16)
  };
  // this wave's chunk of round r of block j
  auto chunk_of = [&](int j, int r) __attribute__((always_inline)) {
    Chunk c;
    if (r < kSw64Rounds) {
      const int* e = entry(j, r, wv);
      c.seg = __builtin_amdgcn_readfirstlane(e[0]);
      c.len = __builtin_amdgcn_readfirstlane(e[1]);
      c.cell = e[3 + lr];
    } else {
      const int q = s_lohi[4 * j] + r * NW + wv;
      const bool has = q < s_lohi[4 * j + 1];
      c.seg = __builtin_amdgcn_readfirstlane(has ? a.ch_seg[q] : -1);
      c.len = __builtin_amdgcn_readfirstlane(has ? a.ch_len[q] : 0);
      const int p0 = has ? a.ch_start[q] : 0;
      c.cell = a.order[(lr < c.len) ? p0 + lr : 0];
    }
    return c;
  };

  // Z rows of a chunk: a row past its length or a load past column d gets an
  // offset past the end of Z and returns zeros (the host checks n d 8 and
  // n K 8 <= kNoRow)
  const __amdgpu_buffer_rsrc_t z_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<double*>(a.Z), (short)0, (int)((unsigned)a.n * (unsigned)d * 8u), 0x00020000);
  const __amdgpu_buffer_rsrc_t r_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      static_cast<void*>(a.R), (short)0, (int)((unsigned)a.n * (unsigned)K * 8u), 0x00020000);
  double z[SM];
  auto load_z = [&](const Chunk& c) __attribute__((always_inline)) {
    const int lr = fresh(lane & 15), lg = fresh(lane >> 4), d = fresh_s(a.d);
    const unsigned zoff = (lr < c.len) ? (unsigned)c.cell * (unsigned)d * 8u : kNoRow;
#pragma unroll
    for (int q = 0; q < SM / 2; ++q) {
      const int col = 8 * q + 2 * lg;
      const doublex2 v = __builtin_bit_cast(
          doublex2, __builtin_amdgcn_raw_buffer_load_b128(
                        z_rsrc, (int)((col < d) ? zoff + 8u * (unsigned)col : 0x80000000u), 0, 0));
      z[2 * q] = v.x;
      z[2 * q + 1] = v.y;
    }
    if constexpr (SM % 2 != 0) {
      const int col = 4 * (SM - 1) + lg;
      z[SM - 1] = __builtin_bit_cast(
          double, __builtin_amdgcn_raw_buffer_load_b64(
                      z_rsrc, (int)((col < d) ? zoff + 8u * (unsigned)col : 0x80000000u), 0, 0));
    }
  };
  // similarities of a chunk's 16 rows; with odd d the value past a row's end
  // (the next row's first) is replaced by zero
  doublex4 acc[NT];
  auto similarities = [&]() __attribute__((always_inline)) {
    const int lr = fresh(lane & 15), lg = fresh(lane >> 4), d = fresh_s(a.d);
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = doublex4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int s = 0; s < SM; ++s) {
      const int c = z64_col<SM>(s, lg);
      const double zv = (c < d) ? z[s] : 0.0;
      __builtin_amdgcn_sched_barrier(0);
      double b[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) b[t] = Ys[c * YS + 16 * t + lr];
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t] = mfma_f64(zv, b[t], acc[t]);
    }
  };

  // objective terms of this lane's rows: k-means, entropy without its row
  // logarithms, and the product of the row sums (its logarithm is their sum)
  double km = 0.0, ent = 0.0, sprod = 1.0;
  int sexp = 0;
  double dO[NT];               // column sums of the wave's current segment
#pragma unroll
  for (int t = 0; t < NT; ++t) dO[t] = 0.0;

  // rows of a chunk (kernels_pen.cuh:27-82): lane holds rows 4 r + lg at
  // columns 16 t + lr.  First the exponentials, in place of the similarities,
  // with each row's sums; then the normalised values.  Neither half keeps more
  // than one value per (row, tile) in registers.
  auto finish = [&](const Chunk& c, int b) __attribute__((always_inline)) {
    const int lr = fresh(lane & 15), lg = fresh(lane >> 4), K = fresh_s(a.K);
    const double term = a.term;
    double s[4], so[4], sl[4];  // sums of e, e (1 - sim), e log pen
#pragma unroll
    for (int r = 0; r < 4; ++r) s[r] = so[r] = sl[r] = 0.0;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      __builtin_amdgcn_sched_barrier(0);  // one tile's exponentials in flight
      const int k = 16 * t + lr;
      double lp = s_lpen[b * K + min(k, K - 1)];
      lp = (k < K) ? lp : -1e5;  // exp64 gives 0
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const double om = 1.0 - acc[t][r];
        const double e = exp64(fma(term, om, lp));
        s[r] += e;
        so[r] = fma(e, om, so[r]);
        sl[r] = fma(e, lp, sl[r]);
        acc[t][r] = e;
        pin(s[r]);
        pin(so[r]);
        pin(sl[r]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    double inv[4];
    unsigned roff[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 4 * r + lg;
      const bool ok = row < c.len;
      const double sr = ok ? sum16(s[r]) : 1.0;
      inv[r] = ok ? 1.0 / sr : 0.0;  // a row past the chunk adds nothing
      km = fma(inv[r], so[r], km);
      ent = fma(inv[r], fma(term, so[r], sl[r]), ent);
      // frexp: the product stays in [0.5, 1)
      const double x = sprod * __builtin_amdgcn_frexp_mant(sr);
      sexp += __builtin_amdgcn_frexp_exp(sr) + __builtin_amdgcn_frexp_exp(x);
      sprod = __builtin_amdgcn_frexp_mant(x);
      pin(km);
      pin(ent);
      pin(sprod);
      const int cell = __shfl(c.cell, row, kWave);
      roff[r] = ok ? (unsigned)cell * (unsigned)K * 8u : kNoRow;
    }
    float eps = 0.f;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      __builtin_amdgcn_sched_barrier(0);
      const unsigned k = 16u * t + (unsigned)lr;
      const unsigned koff = (k < (unsigned)K) ? 8u * k : 0x80000000u;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const double v = acc[t][r] * inv[r];
        dO[t] += v;
        eps += log1p_eps((float)v);
        pin(eps);
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r_rsrc,
                                              (int)(roff[r] + koff), 0, 0);
      }
      pin(dO[t]);
    }
    __builtin_amdgcn_sched_barrier(0);
    ent += (double)eps;
  };
  // the wave's column sums of batch b into the block's sums (the order of the
  // integer adds does not matter)
  auto flush = [&](int b) __attribute__((always_inline)) {
    const int lr = fresh(lane & 15), lg = fresh(lane >> 4), K = fresh_s(a.K);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      double x = dO[t];
      x += __shfl_xor(x, 16, kWave);
      x += __shfl_xor(x, 32, kWave);
      dO[t] = 0.0;
      const int k = 16 * t + lr;
      if (lg == 0 && k < K)
        atomicAdd(&s_dO[b * K + k], (unsigned long long)to_fixed(x, a.scale_blk));
    }
  };

  // O/E update between blocks (clustering.cu:321-347), identical in every
  // workgroup: plus the new rows of block jo (once every contribution has
  // arrived), minus the old rows of block jn; log penalty of jn's batches
  auto update = [&](int jo, int jn) __attribute__((always_inline)) {
    const int tid = fresh(threadIdx.x), K = fresh_s(a.K), B = fresh_s(a.B), BK = B * K;
    const int GB = fresh_s(NTH / a.K), cg = tid / K, ck = tid - cg * K;
    const bool upd = tid < GB * K;
    double* my_o = a.oe + (size_t)wg * 2 * BK + ck;
    double out[kSw64U], in[kSw64U], Or[kSw64U], Er[kSw64U];
#pragma unroll
    for (int u = 0; u < kSw64U; ++u) out[u] = in[u] = 0.0;
    if (upd) {
#pragma unroll
      for (int u = 0; u < kSw64U; ++u) {
        const int p = min(cg + u * GB, B - 1) * K;
        Or[u] = my_o[p];
        Er[u] = my_o[BK + p];
      }
      long long vi[kSw64U];
      if (jn >= 0) {
#pragma unroll
        for (int u = 0; u < kSw64U; ++u)
          vi[u] = a.acc_in[(long long)jn * BK + min(cg + u * GB, B - 1) * K + ck];
      }
      double co = 0.0, ci = 0.0;
      if (jo >= 0) {
        int need[kSw64U];
#pragma unroll
        for (int u = 0; u < kSw64U; ++u) need[u] = a.cnt[jo * B + min(cg + u * GB, B - 1)];
        const long long* src = a.acc_out + (long long)jo * BK + ck;
        long long lo[kSw64U], hi[kSw64U];
        unsigned it = 0;
        while (true) {
#pragma unroll
          for (int u = 0; u < kSw64U; ++u) {
            const long long* p = src + min(cg + u * GB, B - 1) * K;
            lo[u] = load_agent(p);
            hi[u] = load_agent(p + a.rep_stride);
          }
          int short_count = 0;
#pragma unroll
          for (int u = 0; u < kSw64U; ++u)
            short_count |= (int)((lo[u] >> kCountShift) < (long long)need[u]) |
                           (int)((hi[u] >> kCountShift) < (long long)need[u]);
          if (!short_count) break;
          __builtin_amdgcn_s_sleep(1);
          if (++it >= a.spin_limit) {
            // The sums are incomplete: O, E, the objective and the history
            // stay as they were at launch (R does not), since no workgroup
            // is the last to arrive once kSw64GaveUp is set, and the kernels
            // queued behind find the call done.  Waited for, so that it
            // precedes this workgroup's own arrival.
            const int was =
                __hip_atomic_fetch_or(&ctrl->fin, kSw64GaveUp, __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_AGENT) |
                __hip_atomic_fetch_or(&ctrl->pad0, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) |
                __hip_atomic_fetch_or(&ctrl->done, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            asm volatile("" ::"v"(was));
            break;
          }
        }
#pragma unroll
        for (int u = 0; u < kSw64U; ++u) {
          if (cg + u * GB < B) {
            out[u] = (double)(((hi[u] & kValueMask) << kSplitBits) + (lo[u] & kValueMask)) *
                     a.inv_scale_blk;
            co += out[u];
          }
        }
      }
      if (jn >= 0) {
#pragma unroll
        for (int u = 0; u < kSw64U; ++u) {
          if (cg + u * GB < B) {
            in[u] = (double)vi[u] * a.inv_scale_o;
            ci += in[u];
          }
        }
      }
      s_co[tid] = co;
      s_ci[tid] = ci;
    }
    __syncthreads();
    if (upd) {
      double co = 0.0, ci = 0.0;
      for (int g = 0; g < min(GB, B); ++g) {  // groups past B hold nothing
        co += s_co[g * K + ck];
        ci += s_ci[g * K + ck];
      }
      const int bl = (jn >= 0) ? s_lohi[4 * jn + 2] : 0;
      const int bh = (jn >= 0) ? s_lohi[4 * jn + 3] : -1;
#pragma unroll
      for (int u = 0; u < kSw64U; ++u) {
        const int b = cg + u * GB;
        __builtin_amdgcn_sched_barrier(0);
        if (b < B) {
          const double pr = s_pr[b];
          const double o = Or[u] + out[u] - in[u];
          const double e = Er[u] + pr * co - pr * ci;
          my_o[b * K] = o;
          my_o[BK + b * K] = e;
          if (b >= bl && b <= bh) {
            const double denom = a.stabilized ? (o + e + 1.0) : (o + 1.0);
            s_lpen[b * K + ck] = s_th[b] * dlog((e + 1.0) / denom);
          }
        }
      }
    }
    __syncthreads();
  };

  // block 0: its chunks, the penalty without its old rows, first similarities
  int cells[kCellU];
  load_desc(0);
  put_desc(0);
  if (a.nblk > 1) {
    load_desc(1);
    put_desc(1);
  }
  __syncthreads();
  load_cells(0, cells);
  put_cells(0, cells);
  if (a.nblk > 1) {
    load_cells(1, cells);
    put_cells(1, cells);
  }
  __syncthreads();
  Chunk c0 = chunk_of(0, 0);
  load_z(c0);
  update(-1, 0);
  similarities();

  for (int j = 0; j < a.nblk; ++j) {
    const int lo = s_lohi[4 * j], hi = s_lohi[4 * j + 1];
    const bool next = j + 1 < a.nblk, next2 = j + 2 < a.nblk;
    if (next2) load_desc(j + 2);
    for (int q = tid; q < BK; q += NTH) s_dO[q] = 0ull;
    __syncthreads();
    // rounds of NW chunks.  The next chunk's Z rows (of the next round, or of
    // the next block after the last one) are in flight during the epilogue;
    // its similarities follow.
    int qb = -1;
    Chunk c1{-1, 0, 0};
    int r = 0;
    do {
      const bool more = lo + (r + 1) * NW < hi;  // workgroup-uniform
      c1 = Chunk{-1, 0, 0};
      if (more)
        c1 = chunk_of(j, r + 1);
      else if (next)
        c1 = chunk_of(j + 1, 0);
      load_z(c1);
      if (c0.seg >= 0) {  // wave-uniform
        const int b = c0.seg - j * B;
        if (b != qb) {
          if (qb >= 0) flush(qb);
          qb = b;
        }
        finish(c0, b);
      }
      if (!more) break;
      if (c1.seg >= 0) similarities();
      c0 = c1;
      ++r;
    } while (true);
    if (qb >= 0) flush(qb);
    __syncthreads();
    // this workgroup's sums of block j: value words with a count of 1 each
    if (lo < hi) {
      const int bl = s_lohi[4 * j + 2], bh = s_lohi[4 * j + 3];
      for (int q = bl * K + tid; q < (bh + 1) * K; q += NTH) {
        const unsigned long long v = s_dO[q];
        unsigned long long* dst =
            reinterpret_cast<unsigned long long*>(a.acc_out) + (long long)j * BK + q;
        __hip_atomic_fetch_add(dst, (1ull << kCountShift) + (v & ((1ull << kSplitBits) - 1)),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_fetch_add(dst + a.rep_stride, (1ull << kCountShift) + (v >> kSplitBits),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    // while the other workgroups' sums arrive: chunks of block j + 2 and the
    // next chunk's similarities
    if (next2) {
      put_desc(j + 2);
      __syncthreads();
      load_cells(j + 2, cells);
    }
    if (next && c1.seg >= 0) similarities();
    if (next2) put_cells(j + 2, cells);
    c0 = c1;
    update(j, next ? j + 1 : -1);  // its barriers also publish the cells
  }

  // objective terms (kernels_kmeans.cuh:30-95, kernels_clustering.cuh:9-62)
  {
    // the 16 lanes of a row hold the same row sums
    if (lr == 0) ent -= fma((double)sexp, 0.693147180559945309417, dlog(sprod));
    const double k2 = wave_sum(2.0 * km), e2 = wave_sum(ent);
    if (lane == 0) {
      s_obj[wv][0] = k2;
      s_obj[wv][1] = e2;
    }
    __syncthreads();
    if (tid == 0) {
      double k4 = 0.0, e4 = 0.0;
      for (int w = 0; w < NW; ++w) {
        k4 += s_obj[w][0];
        e4 += s_obj[w][1];
      }
      const int rep = wg % kRep;
      const unsigned long long r0 = fixed_add_wait(&a.obj_acc[2 * rep], k4, a.scale_obj);
      const unsigned long long r1 = fixed_add_wait(&a.obj_acc[2 * rep + 1], e4, a.scale_obj);
      asm volatile("" ::"v"(r0 + r1));
    }
  }
  if (!last_to_arrive_of(&ctrl->fin, G, &s_last)) return;

  // last workgroup: O/E, objective, window-3 test (clustering.cu:375-387)
  double div = 0.0;
  if (upd) {
#pragma unroll
    for (int u = 0; u < kSw64U; ++u) {
      const int b = cg + u * GB;
      __builtin_amdgcn_sched_barrier(0);
      if (b < B) {
        const double o = my_o[b * K], e = my_o[BK + b * K];
        a.O[b * K + ck] = o;
        a.E[b * K + ck] = e;
        const double numer = a.stabilized ? (o + e + 1.0) : (o + 1.0);
        div += s_th[b] * o * dlog(numer / (e + 1.0));
      }
    }
  }
  div = block_sum(div, red);
  if (tid == 0) {
    long long qk = 0, qe = 0;
    for (int r = 0; r < kRep; ++r) {
      qk += load_agent(&a.obj_acc[2 * r]);
      qe += load_agent(&a.obj_acc[2 * r + 1]);
    }
    const double obj = (double)qk * a.inv_scale_obj + a.sigma * ((double)qe * a.inv_scale_obj) +
                       a.sigma * div;
    const int nobj = ctrl->n_obj + 1;
    ctrl->n_obj = nobj;
    ctrl->hist[(nobj - 1) & 3] = obj;
    if (a.last_obj) *a.last_obj = obj;
    if (nobj >= 4) {
      double old_s = 0.0, new_s = 0.0;
      for (int w = 0; w < 3; ++w) {
        old_s += ctrl->hist[(nobj - 2 - w) & 3];
        new_s += ctrl->hist[(nobj - 1 - w) & 3];
      }
      if ((old_s - new_s) < a.tol * fabs(old_s)) ctrl->done = 1;
    }
    __hip_atomic_store(&ctrl->fin, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

}  // namespace hz
