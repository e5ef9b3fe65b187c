// Host-side declarations shared by the translation units of libharmony_hip:
// the workspace layout of a job and the launchers of the templated
// matrix-core kernels (each launcher's instantiations compile in a unit of
// their own, so the library builds in parallel).
#pragma once

#include <algorithm>

#include "hz_correct.hpp"
#include "hz_sweep.hpp"
#include "hz_cent64.hpp"
#include "hz_kmeans.hpp"
#include "hz_sweep64.hpp"

namespace hz {

struct Layout {
  int n, d, K, B, bs, esz;
  // several covariates: B counts the groups of cells sharing all levels, BL
  // the levels (rows of O and E), BL0 those of covariate 0; one covariate:
  // C = 1, BL = BL0 = B, glev = nullptr
  int C, BL, BL0;
  const int* glev;
  long long nacc;  // accumulator rows: nblk x BL
  int CT, Kp, DT, Dp;
  int chunk, chunk_p, G, cpw;
  // matrix-core path (FP32 storage)
  int mfma, prec, NT, NU, dP, cent_mfma, Gm, cpwm;
  void* YH;
  void* YL;
  PermDims pd;
  PermDims sd;  // static row chunks (cells grouped by batch)
  PermDims spd; // static phi chunks
  // clustering
  PermBufs pb;
  ChunkTab ct;   // block-order tables of nord iterations (tab_of)
  int nord;
  int* nch_tmp;
  ChunkTab st;
  int* nch_tmp_s;
  ChunkTab sp;
  int* nch_tmp_p;
  long long* acc_in;
  long long* acc_out;  // kRep replicas
  long long* obj_acc;  // kRep x 2
  Ctrl* ctrl;
  Ctrl* ctrl_static;  // never set done: used by the correction pass
  int* counters;      // nblk + 6
  int* swcnt;         // nblk * B * kSweepRep: block-sweep contribution counts
  int Gs = 1;         // workgroups of the streaming centroid pass
  double* oe;         // FP64 sweep: 2 x B x K per workgroup (one per CU)
  void* Ypart;
  double* Yslice;  // kYSlices x K x d: centroid reduction slices
  int* ycnt;       // K arrival counters of the centroid reduction
  void* Y;
  void* YT;
  void* pen;
  // correction
  void* phipart;
  double* Phi;
  long long* rsum;
  void* lam;
  void* Wt;
  double* Wl;  // several covariates: per-level solutions, K x (BL + 1) x d
  size_t bytes;
  double scale_o, scale_obj;
};

// k-steps of the row kernel: f32 4 columns per step, bf16 32 per step
inline int row_sm(const Layout& L) {
  if (L.prec == HZ_PREC_SPLIT_BF16) return (int)ceil_div(L.d, 32);  // 1..4
  const int s = (int)ceil_div(L.d, 4);
  return s <= 4 ? 4 : s <= 8 ? 8 : s <= 13 ? 13 : s <= 16 ? 16 : s <= 25 ? 25 : 32;
}

int prepare_lds(const void* kern, size_t lds);
size_t widen_lds(const void* kern, size_t base, size_t want, long long grid);
int tune_value(int key);
int current_device_index();

// Launchers of the templated matrix-core kernels, one set per precision
// (defined in hz_k_*.hip); the unsuffixed dispatchers pick by L.prec.
int launch_row_mfma_f32(const Layout& L, const RowMArgs& a, int grid, hipStream_t s);
int launch_row_mfma_bf16(const Layout& L, const RowMArgs& a, int grid, hipStream_t s);
// a == nullptr: choose the grid only; HZ_ERR_UNSUPPORTED when not co-resident
int launch_sweep_f32(const Layout& L, const SweepArgs* a, int* G, hipStream_t s);
int launch_sweep_bf16(const Layout& L, const SweepArgs* a, int* G, hipStream_t s);
// several jobs of one kernel shape in one cooperative sweep launch; d_jobs ==
// nullptr: only the co-resident capacity (*cap workgroups) for `lds` bytes
int sweep_multi_f32(const Layout& L, size_t lds, const SweepArgs* d_jobs, const int* d_off,
                    int n_jobs, int G, int* cap, hipStream_t s);
int sweep_multi_bf16(const Layout& L, size_t lds, const SweepArgs* d_jobs, const int* d_off,
                     int n_jobs, int G, int* cap, hipStream_t s);
// FP64 block sweep: a == nullptr chooses the grid only; HZ_ERR_UNSUPPORTED
// (nothing launched) when the shape has no kernel or is not co-resident
int launch_sweep64(const Layout& L, const Sweep64Args* a, int* G, hipStream_t s);
// FP64 centroid pass in natural order (fills in tg and rows); *grid: the number
// of partials written, at most max_grid.  HZ_ERR_UNSUPPORTED (nothing launched)
// above 128 clusters or columns
int launch_cent64(const Cent64Args& a, int* grid, int max_grid, hipStream_t s);
// Lloyd assignment and partial sums; HZ_ERR_UNSUPPORTED (nothing launched)
// above 128 clusters or columns or where the LDS does not hold them
int launch_kmeans_assign(const KmMArgs<float>& a, int grid, hipStream_t s);
int launch_kmeans_assign(const KmMArgs<double>& a, int grid, hipStream_t s);
size_t sweep_lds_f32(const Layout& L);
size_t sweep_lds_bf16(const Layout& L);
int launch_cent_stream_f32(const Layout& L, const CentSArgs* jobs, const int* off, int n_jobs,
                           int grid, hipStream_t s);
int launch_cent_stream_bf16(const Layout& L, const CentSArgs* jobs, const int* off, int n_jobs,
                            int grid, hipStream_t s);
int launch_cent_mfma_f32(const Layout& L, const CentMArgs& a, int grid, hipStream_t s);
int launch_cent_mfma_bf16(const Layout& L, const CentMArgs& a, int grid, hipStream_t s);
// FP32 correction apply on matrix cores; HZ_ERR_UNSUPPORTED (nothing
// launched) when its LDS does not fit
int launch_apply_mfma(const Layout& L, const ApplyMArgs& a, int grid, hipStream_t s);
// Cooperative launch of a kernel that takes one argument struct; waits, like a
// block sweep, for the previous grid whose workgroups depend on each other.
// HZ_ERR_UNSUPPORTED when the runtime refuses the launch (not launched then)
int chained_cooperative(hipStream_t s, const void* kern, int grid, int block, void* arg);
void mark_sweep_broken();
bool sweep_broken();

// Workgroups of a block sweep that may use up to `cap`: as many as give every
// wave the same number of chunks in the fewest rounds.  More would not shorten
// a block (the rounds stay), but every workgroup adds to and reads the block's
// sums: one round of 320 chunks (100k cells, 8 batches) takes 191 us per sweep
// on 81-96 workgroups, 228 us on 256; 1310 chunks of 5 batches (417k cells)
// 2 rounds either way, 297 us on 192, 401 us on 256.  Below about 40 the sums'
// exchange no longer costs, and a chunk runs faster on a CU of its own (3k
// cells: 163 us on 24-64, 168 us on 4-16; 10k: 140-146 us on 24-48, 180 us on 8).
// The fixed-point sums do not depend on it.  (sweep_readers adds workgroups
// without rows where there are many batches.)
inline int sweep_wgs(const Layout& L, int cap, int nw = kBlock / kWave) {
  const long long chunks = ceil_div(L.bs, L.chunk) + L.B;  // each batch's last chunk is partial
  const long long rounds = ceil_div(chunks, (long long)nw * cap);  // nw: waves of a workgroup
  return (int)std::min<long long>(cap, std::max<long long>(40, ceil_div(chunks, nw * rounds)));
}

// Workgroups without rows beside the `wgs` with them in an FP32 sweep.  Above
// eight batches per thread a block's old-row deltas are not held in registers:
// they are read when the block's rows are done, from HBM unless another
// workgroup of the XCD has read them before.  One without rows on every XCD
// (workgroups go to the eight in turn) is always ahead.  us per sweep, 100
// clusters, with and without: 100k cells x 24 batches 265 and 296, 200k x 32 306
// and 338, 1M x 32 (split-BF16) 460 and 481; 256 workgroups take 265, 305, 465.
inline int sweep_readers(const Layout& L, int wgs, int cap) {
  constexpr int kXcd = 8;
  return L.B > kSweepInRegs * std::max(1, kBlock / L.K) && wgs + kXcd <= cap ? kXcd : 0;
}

inline int launch_row_mfma(const Layout& L, const RowMArgs& a, int grid, hipStream_t s) {
  return L.prec == HZ_PREC_SPLIT_BF16 ? launch_row_mfma_bf16(L, a, grid, s)
                                      : launch_row_mfma_f32(L, a, grid, s);
}
inline int launch_sweep(const Layout& L, const SweepArgs* a, int* G, hipStream_t s) {
  return L.prec == HZ_PREC_SPLIT_BF16 ? launch_sweep_bf16(L, a, G, s) : launch_sweep_f32(L, a, G, s);
}
inline int sweep_multi(const Layout& L, size_t lds, const SweepArgs* d_jobs, const int* d_off,
                       int n_jobs, int G, int* cap, hipStream_t s) {
  return L.prec == HZ_PREC_SPLIT_BF16 ? sweep_multi_bf16(L, lds, d_jobs, d_off, n_jobs, G, cap, s)
                                      : sweep_multi_f32(L, lds, d_jobs, d_off, n_jobs, G, cap, s);
}
inline size_t sweep_lds_of(const Layout& L) {
  return L.prec == HZ_PREC_SPLIT_BF16 ? sweep_lds_bf16(L) : sweep_lds_f32(L);
}
// n_jobs jobs of L's kernel shape, arguments and workgroup offsets on the device
inline int launch_cent_stream_multi(const Layout& L, const CentSArgs* jobs, const int* off,
                                    int n_jobs, int grid, hipStream_t s) {
  return L.prec == HZ_PREC_SPLIT_BF16 ? launch_cent_stream_bf16(L, jobs, off, n_jobs, grid, s)
                                      : launch_cent_stream_f32(L, jobs, off, n_jobs, grid, s);
}
inline int launch_cent_stream(const Layout& L, const CentSArgs& a, int grid, hipStream_t s) {
  return launch_cent_stream_multi(L, &a, nullptr, 1, grid, s);
}
inline int launch_cent_mfma(const Layout& L, const CentMArgs& a, int grid, hipStream_t s) {
  return L.prec == HZ_PREC_SPLIT_BF16 ? launch_cent_mfma_bf16(L, a, grid, s)
                                      : launch_cent_mfma_f32(L, a, grid, s);
}

}  // namespace hz
