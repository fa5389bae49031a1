// Prioritised replay on the device: the step between V-trace and the MinGRU BPTT.
//
//   ph_seg_l1       sum_t |adv(e,t)| per segment                         (k_adv_l1, puffercuda.cu:311-312)
//   ph_prio_sample  prioritised segment draws + importance weights       (puffercuda.cu:400-470; CPU twin
//                                                                          pufferffi.c:1094-1125)
//   ph_mb_gather    minibatch columns, timestep-major, adv normalised    (puffercuda.cu:472-502; CPU twin
//                                                                          pufferffi.c:1126-1200)
//   ph_mb_iterate   value/ratio of the sampled segments from the BPTT    (puffercuda.cu:503-511)
//
// Design: the reference chains seven launches for the sampler (weights, a one-block sum, a 64-chunk
// single-thread scan, its combine and add, the draws). Here it is one for a few segments and draws, else two: the
// segment weights, then blocks that each form the fixed-tree sum and the cumulative table in their own LDS and
// take a share of the draws (one workgroup for them once the table outgrows LDS). The gather is one pass that also produces per-block
// (count, mean, M2) partials; the normalising kernel's blocks merge them in block order (Chan et al.'s
// pairwise update), so mean and std cost no extra pass over the columns. Segment-major columns pass
// through LDS tiles of 16 segments x 64 steps, so that both the segment rows and the timestep-major
// minibatch are read and written in runs. The iterate writes the last draw of a segment: found by comparing the
// draws in each block, or for many draws and time-major columns through a last-writer table that the second
// launch leaves zeroed.
//
// Every reduction here has a fixed order, so results are reproducible run to run. They are not
// bit-identical to the CPU twins, whose sums are sequential: mean, std, the probability normaliser
// and the cumulative table agree to rounding, and device exp/log agree with the host's to an ulp. A
// draw whose uniform lies within that rounding of a cumulative boundary can therefore pick the
// neighbouring segment; the reference's own device sampler has the same property.
#include <cmath>

#include "common.hpp"
#include "kernels.hpp"
#include "routes.hpp"

// The formulas below execute in the order written (no fused multiply-add), as in the CPU twins.
#pragma clang fp contract(off)

namespace ph {
namespace {

constexpr int kPsThreads = 1024;
constexpr long kPsLdsCum = 8192;  // cumulative table held in LDS up to this many segments (64 KiB)
constexpr int kPsDraws = 128;     // draws per block of the LDS sampler
constexpr int kGaThreads = 256;
constexpr int kGaPer = 4;         // minibatch elements per gather thread (256 blocks at 4096 x 64)
constexpr int kGaBlock = kGaThreads * kGaPer;
constexpr int kSm = 16, kSt = 64;    // tile of segment-major columns: segments x steps
constexpr int kSp = kSt + 1;         // its LDS pitch (a step of 16 segments hits distinct banks)
inline bool sm_tiles(const ph_replay_cols& c) { return gather_tiled(c.time_major, (long)c.T); }

// ---- per-segment |adv| sums ------------------------------------------------------------------------
// t ascending, f64 accumulation (the reference's order). One thread per segment: time-major columns
// (coalesced across the segment threads) and the segment-major ones seg_l1_tiled leaves.
template <typename R, bool TM>
__global__ void __launch_bounds__(256) k_seg_l1(const R* __restrict__ adv, long N, int T, double* __restrict__ L1) {
  const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= N) return;
  double s = 0.0;
#pragma unroll 8
  for (int t = 0; t < T; t++) s += fabs((double)adv[TM ? (long)t * N + e : e * T + t]);
  L1[e] = s;
}
// Segment-major: a block's 16 segments arrive 64 steps at a time in 64-wide runs (a thread per segment reads T
// elements apart from its neighbours, on N / 64 wavefronts), and one lane per segment adds its row out of
// LDS in order. 8192x64 f64: 5.1 -> 3.0 us.
template <typename R>
__global__ void __launch_bounds__(256) k_seg_l1_sm(const R* __restrict__ adv, long N, int T, double* __restrict__ L1) {
  __shared__ double tl[kSm][kSp];
  const long e0 = (long)blockIdx.x * kSm;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  double v[kSm / 4];
  const auto load = [&](int t0) {
#pragma unroll
    for (int i = 0; i < kSm / 4; i++) {
      const long e = e0 + w + 4 * i;
      v[i] = e < N && t0 + lane < T ? fabs((double)adv[e * T + t0 + lane]) : 0.0;
    }
  };
  load(0);
  double s = 0.0;
  for (int t0 = 0; t0 < T; t0 += kSt) {
#pragma unroll
    for (int i = 0; i < kSm / 4; i++) tl[w + 4 * i][lane] = v[i];
    __syncthreads();
    if (t0 + kSt < T) load(t0 + kSt);
    if (threadIdx.x < kSm) {
      const int n = T - t0 < kSt ? T - t0 : kSt;
#pragma unroll 16
      for (int t = 0; t < n; t++) s += tl[threadIdx.x][t];
    }
    __syncthreads();
  }
  if (threadIdx.x < kSm && e0 + threadIdx.x < N) L1[e0 + threadIdx.x] = s;
}

// ---- prioritised sampler ---------------------------------------------------------------------------
// Thread i of a 1024-thread block owns the contiguous segment chunk [i*R, min(N, (i+1)*R)).
//   w[e]   = exp(alpha * log(L1[e] + 1e-12))
//   p[e]   = (w[e] + 1e-6) / (sum w + 1e-6)            (sum: per-chunk sequential, then a fixed tree)
//   cum[e] = chunk-local running sum of p + the sum of the earlier chunks (fixed-tree scan)
//   draw i: z = splitmix64 finaliser of rng + (i+1)*GOLD; u = (z >> 11) / 2^53 * total;
//           idx = first e with cum[e] >= u (N-1 if none); mp[i] = exp(-beta * log(N * p[idx] + 1e-12))
// Past a few segments and draws (prio_one_block) the f64 exponentials and logarithms of the weights and the draws
// are what takes the time in one workgroup, so they are spread over the chip: a kernel of weights, then (N up to
// kPsLdsCum) blocks of kPsDraws draws that each form the table from the weights in their LDS, the same
// operations in the same order in every block.
// 4096 segments, 4096 draws: 21.9 us in one workgroup, 10.1 in the two launches.
__device__ __forceinline__ double prio_p(double w, double denom) { return (w + 1e-6) / denom; }

__device__ __forceinline__ double prio_weight(double l1, double alpha) { return exp(alpha * log(l1 + 1e-12)); }

__global__ void __launch_bounds__(256) k_prio_weights(const double* __restrict__ L1, long N, double alpha,
                                                      double* __restrict__ w) {
  const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e < N) w[e] = prio_weight(L1[e], alpha);
}

// The cumulative table of the block's threads into cum; returns the total. red: kPsThreads doubles.
__device__ inline double prio_table(const double* w, long N, double* cum, double* red, double& denom) {
  const int tid = threadIdx.x;
  const long R = (N + kPsThreads - 1) / kPsThreads;
  const long lo = (long)tid * R < N ? (long)tid * R : N;
  const long hi = lo + R < N ? lo + R : N;
  double s = 0.0;
  for (long e = lo; e < hi; e++) s += w[e];
  red[tid] = s;
  __syncthreads();
  for (int st = kPsThreads / 2; st > 0; st >>= 1) {
    if (tid < st) red[tid] += red[tid + st];
    __syncthreads();
  }
  denom = red[0] + 1e-6;
  __syncthreads();
  double c = 0.0;
  for (long e = lo; e < hi; e++) {
    c += prio_p(w[e], denom);
    cum[e] = c;
  }
  // inclusive scan of the chunk totals (Hillis-Steele, fixed order)
  red[tid] = c;
  __syncthreads();
  for (int off = 1; off < kPsThreads; off <<= 1) {
    const double v = tid >= off ? red[tid - off] : 0.0;
    __syncthreads();
    if (tid >= off) red[tid] += v;
    __syncthreads();
  }
  const double carry = tid > 0 ? red[tid - 1] : 0.0;
  const double total = red[kPsThreads - 1];
  if (tid > 0)
    for (long e = lo; e < hi; e++) cum[e] += carry;
  __syncthreads();
  return total;
}

__device__ inline void prio_draw(long i, const double* cum, const double* w, long N, double total, double denom,
                                 double beta, unsigned long long rng, int* __restrict__ seg, double* __restrict__ mp) {
  unsigned long long z = rng + (unsigned long long)(i + 1) * 0x9E3779B97F4A7C15ULL;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
  z = z ^ (z >> 31);
  const double u = (double)(z >> 11) / 9007199254740992.0 * total;
  long L = 0, Rb = N;
  while (L < Rb) {
    const long mid = (L + Rb) >> 1;
    if (cum[mid] >= u) Rb = mid;
    else L = mid + 1;
  }
  const long idx = L < N ? L : N - 1;
  seg[i] = (int)idx;
  mp[i] = exp((-beta) * log((double)N * prio_p(w[idx], denom) + 1e-12));
}

// N up to kPsLdsCum: block b takes draws [b * kPsDraws, (b + 1) * kPsDraws).
__global__ void __launch_bounds__(kPsThreads) k_prio_draws(const double* __restrict__ w, long N, long B, double beta,
                                                           unsigned long long rng, int* __restrict__ seg,
                                                           double* __restrict__ mp) {
  __shared__ double red[kPsThreads];
  __shared__ double cum[kPsLdsCum];
  static_assert((kPsThreads + kPsLdsCum) * 8 <= kMaxLdsBytes, "LDS budget");
  double denom;
  const double total = prio_table(w, N, cum, red, denom);
  const long i = (long)blockIdx.x * kPsDraws + threadIdx.x;
  if (threadIdx.x < kPsDraws && i < B) prio_draw(i, cum, w, N, total, denom, beta, rng, seg, mp);
}

// prio_one_block: weights, table and draws in one launch of one workgroup.
constexpr long kPsOne = 2048;
__global__ void __launch_bounds__(kPsThreads) k_prio_one(const double* __restrict__ L1, long N, long B, double alpha,
                                                         double beta, unsigned long long rng, int* __restrict__ seg,
                                                         double* __restrict__ mp) {
  __shared__ double red[kPsThreads];
  __shared__ double w[kPsOne], cum[kPsOne];
  static_assert((kPsThreads + 2 * kPsOne) * 8 <= kMaxLdsBytes, "LDS budget");
  for (long e = threadIdx.x; e < N; e += kPsThreads) w[e] = prio_weight(L1[e], alpha);
  __syncthreads();
  double denom;
  const double total = prio_table(w, N, cum, red, denom);
  for (long i = threadIdx.x; i < B; i += kPsThreads) prio_draw(i, cum, w, N, total, denom, beta, rng, seg, mp);
}

// More segments: one workgroup, the table in memory.
__global__ void __launch_bounds__(kPsThreads) k_prio_sample(const double* __restrict__ w, long N, long B, double beta,
                                                            unsigned long long rng, double* cum,
                                                            int* __restrict__ seg, double* __restrict__ mp) {
  __shared__ double red[kPsThreads];
  double denom;
  const double total = prio_table(w, N, cum, red, denom);
  for (long i = threadIdx.x; i < B; i += kPsThreads) prio_draw(i, cum, w, N, total, denom, beta, rng, seg, mp);
}

// ---- minibatch gather ------------------------------------------------------------------------------
// Chan et al.'s pairwise merge of (count, mean, M2) summaries.
__device__ inline void chan_merge(double& n, double& m, double& M2, double nb, double mb, double M2b) {
  if (nb == 0.0) return;
  if (n == 0.0) {
    n = nb; m = mb; M2 = M2b;
    return;
  }
  const double nn = n + nb, d = mb - m;
  m = m + d * (nb / nn);
  M2 = M2 + M2b + d * d * (n * nb / nn);
  n = nn;
}

// The block's (count, mean, M2) of its threads' av[0 .. cnt) (sum s) into part, by fixed-tree sums.
__device__ inline void block_moments(double (&sh)[3][kGaThreads], double s, int cnt, const double (&av)[kGaPer],
                                     double* __restrict__ part) {
  const int tid = threadIdx.x;
  sh[0][tid] = s;
  sh[1][tid] = (double)cnt;
  __syncthreads();
  for (int st = kGaThreads / 2; st > 0; st >>= 1) {
    if (tid < st) {
      sh[0][tid] += sh[0][tid + st];
      sh[1][tid] += sh[1][tid + st];
    }
    __syncthreads();
  }
  const double bn = sh[1][0];
  const double bm = bn > 0.0 ? sh[0][0] / bn : 0.0;
  __syncthreads();
  double q = 0.0;
#pragma unroll
  for (int k = 0; k < kGaPer; k++)
    if (k < cnt) {
      const double d = av[k] - bm;
      q += d * d;
    }
  sh[2][tid] = q;
  __syncthreads();
  for (int st = kGaThreads / 2; st > 0; st >>= 1) {
    if (tid < st) sh[2][tid] += sh[2][tid + st];
    __syncthreads();
  }
  if (tid == 0) {
    part[0] = bn;
    part[1] = bm;
    part[2] = sh[2][0];
  }
}

// Output element j = t*B + bi (timestep-major) reads source row e = seg[bi] at step t:
//   act (K wide, truncated to an integer) | adv (raw here) | ret = adv + value | old = logp |
//   term = term > 0.5 ? 1 : 0 | ov = value
// An index outside [0, N) yields NaN columns for that row (the sampler never produces one).
// Each block also reduces its raw adv values to (count, mean, M2) in part; the normalising kernel (or k_mb_stats,
// past gather_folds) merges the blocks in index order into stats = [mean, std] (population std).
template <typename R, bool TM>
__global__ void __launch_bounds__(kGaThreads) k_mb_gather(
    const R* __restrict__ adv, const R* __restrict__ value, const R* __restrict__ act,
    const R* __restrict__ logp, const R* __restrict__ term, long N, int T, int K,
    const int* __restrict__ seg, long B, R* __restrict__ out, double* __restrict__ part) {
  __shared__ double sh[3][kGaThreads];
  const long n = B * T;
  const int tid = threadIdx.x;
  R* oact = out;
  R* oadv = out + (long)K * n;
  R* oret = oadv + n;
  R* oold = oret + n;
  R* oterm = oold + n;
  R* oov = oterm + n;
  const R qnan = (R)__builtin_nan("");
  // Workgroups are dispatched round-robin over the 8 XCDs; XCD x takes the contiguous run of
  // logical blocks [start_x, start_x + count_x), i.e. a contiguous range of steps t, so its L2 holds
  // about an eighth of the source rows instead of all of them.
  const unsigned q8 = gridDim.x / 8, r8 = gridDim.x % 8, x8 = blockIdx.x % 8;
  const unsigned lb = x8 * q8 + (x8 < r8 ? x8 : r8) + blockIdx.x / 8;
  double av[kGaPer];
  int cnt = 0;
  double s = 0.0;
#pragma unroll
  for (int k = 0; k < kGaPer; k++) {
    const long j = (long)lb * kGaBlock + (long)k * kGaThreads + tid;
    av[k] = 0.0;
    if (j < n) {
      const long t = j / B, bi = j - t * B;
      const long e = seg[bi];
      if (e >= 0 && e < N) {
        const long si = TM ? t * N + e : e * T + t;
        const R a = adv[si], v = value[si];
        for (int h = 0; h < K; h++) oact[j * K + h] = (R)trunc((double)act[si * K + h]);
        oadv[j] = a;
        oret[j] = a + v;
        oold[j] = logp[si];
        oterm[j] = term[si] > (R)0.5 ? (R)1 : (R)0;
        oov[j] = v;
        av[k] = (double)a;
        s += av[k];
      } else {
        for (int h = 0; h < K; h++) oact[j * K + h] = qnan;
        oadv[j] = qnan; oret[j] = qnan; oold[j] = qnan; oterm[j] = qnan; oov[j] = qnan;
        av[k] = (double)qnan;
        s += av[k];
      }
      cnt++;
    }
  }
  block_moments(sh, s, cnt, av, part + 3 * (size_t)lb);
}

// Segment-major: a block's tile is draws [16 b, 16 b + 16) x 64 steps. The segments' rows load in 64-wide
// runs, turn in LDS, and the columns store in 16-wide runs of the timestep-major output (a thread per output
// element reads T elements apart from its neighbours). 4096 draws x 64 f64: 12.9 -> 10.1 us.
template <typename R>
__global__ void __launch_bounds__(kGaThreads) k_mb_gather_sm(
    const R* __restrict__ adv, const R* __restrict__ value, const R* __restrict__ act,
    const R* __restrict__ logp, const R* __restrict__ term, long N, int T, int K,
    const int* __restrict__ seg, long B, R* __restrict__ out, double* __restrict__ part) {
  __shared__ R tl[4][kSm][kSp];
  __shared__ double sh[3][kGaThreads];
  const long n = B * T;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const unsigned tiles = (unsigned)((T + kSt - 1) / kSt);
  const long b0 = (long)(blockIdx.x / tiles) * kSm;
  const int t0 = (int)(blockIdx.x % tiles) * kSt, t = t0 + lane;
  const R qnan = (R)__builtin_nan("");
  double av[kGaPer];
  int cnt = 0;
  double s = 0.0;
  bool in[kGaPer], ok[kGaPer];
  long si[kGaPer];
#pragma unroll
  for (int k = 0; k < kGaPer; k++) {  // row w + 4 k of the tile, step t
    const long bi = b0 + w + 4 * k;
    in[k] = bi < B && t < T;
    const long e = bi < B ? seg[bi] : -1;
    ok[k] = in[k] && e >= 0 && e < N;
    si[k] = e * T + t;
  }
  R c[4][kGaPer], x[kGaPer];
#pragma unroll
  for (int k = 0; k < kGaPer; k++) {
    c[0][k] = ok[k] ? adv[si[k]] : qnan;
    c[1][k] = ok[k] ? value[si[k]] : qnan;
    c[2][k] = ok[k] ? logp[si[k]] : qnan;
    c[3][k] = !ok[k] ? qnan : term[si[k]] > (R)0.5 ? (R)1 : (R)0;
    x[k] = ok[k] ? act[si[k] * K] : qnan;
  }
#pragma unroll
  for (int k = 0; k < kGaPer; k++) {
    av[k] = 0.0;
    if (in[k]) {  // rows ascend with k, so the rows in range come first
      av[k] = (double)c[0][k];
      s += av[k];
      cnt++;
    }
#pragma unroll
    for (int q = 0; q < 4; q++) tl[q][w + 4 * k][lane] = c[q][k];
  }
  __syncthreads();
  R* oadv = out + (long)K * n;
  const int ob = tid & (kSm - 1), ot = tid / kSm;
  const long bi = b0 + ob;
  if (bi < B)
#pragma unroll
    for (int k = 0; k < kSt * kSm / kGaThreads; k++) {
      const int u = ot + k * (kGaThreads / kSm);
      if (t0 + u >= T) break;
      const long j = (long)(t0 + u) * B + bi;
      const R a = tl[0][ob][u], v = tl[1][ob][u];
      oadv[j] = a;
      oadv[j + n] = a + v;
      oadv[j + 2 * n] = tl[2][ob][u];
      oadv[j + 3 * n] = tl[3][ob][u];
      oadv[j + 4 * n] = v;
    }
  for (int h = 0; h < K; h++) {  // action components, one at a time through the first tile
    if (h > 0)
#pragma unroll
      for (int k = 0; k < kGaPer; k++) x[k] = ok[k] ? act[si[k] * K + h] : qnan;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kGaPer; k++) tl[0][w + 4 * k][lane] = (R)trunc((double)x[k]);
    __syncthreads();
    if (bi < B)
#pragma unroll
      for (int k = 0; k < kSt * kSm / kGaThreads; k++) {
        const int u = ot + k * (kGaThreads / kSm);
        if (t0 + u >= T) break;
        out[((long)(t0 + u) * B + bi) * K + h] = tl[0][ob][u];
      }
  }
  block_moments(sh, s, cnt, av, part + 3 * (size_t)blockIdx.x);
}

// Thread i folds the gather blocks i, i+256, ... in order, then a fixed tree over the threads: mean and std in
// every thread. Launched after the gather, whose partials the launch boundary orders.
__device__ inline void fold_moments(const double* __restrict__ part, unsigned G, double& mean, double& std) {
  __shared__ double sh[3][kGaThreads];
  const int tid = threadIdx.x;
  double mn = 0.0, mm = 0.0, mq = 0.0;
  for (unsigned b = tid; b < G; b += kGaThreads)
    chan_merge(mn, mm, mq, part[3 * (size_t)b], part[3 * (size_t)b + 1], part[3 * (size_t)b + 2]);
  sh[0][tid] = mn;
  sh[1][tid] = mm;
  sh[2][tid] = mq;
  __syncthreads();
  for (int st = kGaThreads / 2; st > 0; st >>= 1) {
    if (tid < st) {
      double a0 = sh[0][tid], a1 = sh[1][tid], a2 = sh[2][tid];
      chan_merge(a0, a1, a2, sh[0][tid + st], sh[1][tid + st], sh[2][tid + st]);
      sh[0][tid] = a0;
      sh[1][tid] = a1;
      sh[2][tid] = a2;
    }
    __syncthreads();
  }
  const double nt = sh[0][0] > 0.0 ? sh[0][0] : 1.0;
  mean = sh[1][0];
  std = sqrt(sh[2][0] / nt);
}
__global__ void __launch_bounds__(kGaThreads) k_mb_stats(const double* __restrict__ part, unsigned G,
                                                         double* __restrict__ stats) {
  double mean, std;
  fold_moments(part, G, mean, std);
  if (threadIdx.x == 0) {
    stats[0] = mean;
    stats[1] = std;
  }
}

// adv[j] = mp[bi] * (adv[j] - mean) / (std + 1e-8), j = t*B + bi (mp NULL: weight 1). FOLD: every block merges
// the gather's partials itself (gather_folds: the merge costs less than a launch of one block), and the first
// writes stats; else stats are given.
template <typename R, bool FOLD>
__global__ void __launch_bounds__(kGaThreads) k_mb_normalize(R* __restrict__ adv, long B, long n,
                                                             const double* __restrict__ mp,
                                                             const double* __restrict__ part, unsigned G,
                                                             double* __restrict__ stats) {
  R a[kGaPer];
  double w[kGaPer];
  const long j0 = (long)blockIdx.x * kGaBlock + threadIdx.x;
#pragma unroll
  for (int k = 0; k < kGaPer; k++) {
    const long j = j0 + (long)k * kGaThreads;
    a[k] = (R)0;
    w[k] = 1.0;
    if (j < n) {
      a[k] = adv[j];
      if (mp) w[k] = mp[n <= 0xffffffffL ? (long)((unsigned)j % (unsigned)B) : j % B];
    }
  }
  double mean, std;
  if constexpr (FOLD) {
    fold_moments(part, G, mean, std);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      stats[0] = mean;
      stats[1] = std;
    }
  } else {
    mean = stats[0];
    std = stats[1];
  }
#pragma unroll
  for (int k = 0; k < kGaPer; k++) {
    const long j = j0 + (long)k * kGaThreads;
    if (j < n) adv[j] = (R)(w[k] * ((double)a[k] - mean) / (std + 1e-8));
  }
}

// ---- value / ratio iterate -------------------------------------------------------------------------
// Pass 1: lw[e] = max over the draws bi of segment e of (bi + 1). The table is all zero between
// calls: pass 2 clears every entry pass 1 set.
__global__ void __launch_bounds__(256) k_mb_lastw(const int* __restrict__ seg, long B, long N, int* lw) {
  const long bi = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (bi >= B) return;
  const int e = seg[bi];
  if (e >= 0 && e < N) atomicMax(&lw[e], (int)(bi + 1));
}

// Pass 2: one wavefront per draw bi, lanes over t. Only the last draw of a segment (the writer an
// in-order loop over bi leaves in place) stores ratio = exp(newlp - logp) and value = newval, then
// clears the table entry. A draw that reads the entry after the clear sees 0, which matches no draw.
template <typename R, bool TM>
__global__ void __launch_bounds__(256) k_mb_iterate(R* __restrict__ value, R* __restrict__ ratio,
                                                    const R* __restrict__ logp,
                                                    const float* __restrict__ newlp,
                                                    const float* __restrict__ newval,
                                                    const int* __restrict__ seg, long B, long N, int T,
                                                    int* lw) {
  const long bi = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (bi >= B) return;
  const int e = seg[bi];
  if (e < 0 || e >= N) return;
  if (lw[e] != (int)(bi + 1)) return;
  for (int t = lane; t < T; t += 64) {
    const long si = TM ? (long)t * N + e : (long)e * T + t;
    const long os = (long)t * B + bi;
    ratio[si] = (R)exp((double)newlp[os] - (double)logp[si]);
    value[si] = (R)newval[os];
  }
  if (lane == 0) lw[e] = 0;
}

// Segment-major, iterate_tiled: one launch, a block per 16 draws x 64 steps. It compares its draws with every later
// draw (a draw whose segment is drawn again is not its last writer) and turns the timestep-major inputs in LDS, so that a
// row's stores are 64-wide runs. The comparison runs while the tile's loads are in flight.
template <typename R>
__global__ void __launch_bounds__(256) k_mb_iterate_sm(R* __restrict__ value, R* __restrict__ ratio,
                                                       const R* __restrict__ logp, const float* __restrict__ newlp,
                                                       const float* __restrict__ newval, const int* __restrict__ seg,
                                                       long B, long N, int T) {
  __shared__ float lp[kSm][kSp], nv[kSm][kSp];
  __shared__ int es[kSm];
  __shared__ unsigned again;  // bit k: draw b0 + k is not its segment's last
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const unsigned tiles = (unsigned)((T + kSt - 1) / kSt);
  const long b0 = (long)(blockIdx.x / tiles) * kSm;
  const int t0 = (int)(blockIdx.x % tiles) * kSt;
  if (tid < kSm) es[tid] = b0 + tid < B ? seg[b0 + tid] : -1;
  if (tid == 0) again = 0u;
  const int ob = tid & (kSm - 1), ot = tid / kSm;
  constexpr int kPer = kSt * kSm / 256;
  float xl[kPer], xv[kPer];
#pragma unroll
  for (int k = 0; k < kPer; k++) {  // a step or draw past the end re-reads the last
    const long os = (long)min(t0 + ot + k * (256 / kSm), T - 1) * B + min(b0 + ob, B - 1);
    xl[k] = newlp[os];
    xv[k] = newval[os];
  }
  __syncthreads();
  int e[kSm];
#pragma unroll
  for (int k = 0; k < kSm; k++) e[k] = es[k];
  unsigned hit = 0u;
  if (tid < kSm)
#pragma unroll
    for (int k = 0; k < kSm; k++) hit |= (unsigned)(k < tid && es[tid] == e[k]) << k;
  constexpr int kAhead = 8;  // loads in flight per thread
  for (long j = b0 + kSm + tid; j < B; j += kAhead * 256) {
    int o[kAhead];
#pragma unroll
    for (int i = 0; i < kAhead; i++) o[i] = j + i * 256 < B ? seg[j + i * 256] : -1;
#pragma unroll
    for (int i = 0; i < kAhead; i++)
#pragma unroll
      for (int k = 0; k < kSm; k++) hit |= (unsigned)(o[i] == e[k]) << k;
  }
  if (hit) atomicOr(&again, hit);
#pragma unroll
  for (int k = 0; k < kPer; k++) {
    lp[ob][ot + k * (256 / kSm)] = xl[k];
    nv[ob][ot + k * (256 / kSm)] = xv[k];
  }
  __syncthreads();
  if (t0 + lane < T)
#pragma unroll
    for (int k = 0; k < kSm / 4; k++) {
      const int r = w + 4 * k;
      if (es[r] < 0 || es[r] >= N || (again >> r & 1u)) continue;
      const long si = (long)es[r] * T + t0 + lane;
      ratio[si] = (R)exp((double)lp[r][lane] - (double)logp[si]);
      value[si] = (R)nv[r][lane];
    }
}

int check_cols(const ph_replay_cols* c, const char* who) {
  PH_REQUIRE(c, "%s: null column descriptor", who);
  PH_REQUIRE(c->dtype == PH_F32 || c->dtype == PH_F64, "%s: dtype must be PH_F32 or PH_F64", who);
  PH_REQUIRE(c->N > 0 && c->N <= 0x7fffffffL && c->T > 0 && c->T <= 0x7fffffffL,
             "%s: N=%zu T=%zu out of range", who, c->N, c->T);
  return PH_OK;
}

}  // namespace

int seg_l1(const ph_replay_cols& c, double* L1, hipStream_t st) {
  const long N = (long)c.N;
  const int T = (int)c.T;
  const unsigned g = ceil_div(c.N, 256), gs = ceil_div(c.N, kSm);
  const bool tiles = seg_l1_tiled(c.dtype == PH_F64, c.time_major, N, T);
  if (c.dtype == PH_F64) {
    if (tiles) k_seg_l1_sm<double><<<gs, 256, 0, st>>>((const double*)c.adv, N, T, L1);
    else if (c.time_major) k_seg_l1<double, true><<<g, 256, 0, st>>>((const double*)c.adv, N, T, L1);
    else k_seg_l1<double, false><<<g, 256, 0, st>>>((const double*)c.adv, N, T, L1);
  } else {
    if (tiles) k_seg_l1_sm<float><<<gs, 256, 0, st>>>((const float*)c.adv, N, T, L1);
    else if (c.time_major) k_seg_l1<float, true><<<g, 256, 0, st>>>((const float*)c.adv, N, T, L1);
    else k_seg_l1<float, false><<<g, 256, 0, st>>>((const float*)c.adv, N, T, L1);
  }
  PH_LAUNCH_CHECK();
  return PH_OK;
}

int prio_sample(const double* L1, size_t N, size_t B, double alpha, double beta, uint64_t rng, int* seg,
                double* mp, hipStream_t st) {
  PH_REQUIRE(N > 0 && N <= 0x7fffffffUL, "prio_sample: N=%zu out of range", N);
  PH_REQUIRE(B <= 0x7fffffffUL, "prio_sample: %zu draws out of range", B);
  if (B == 0) return PH_OK;
  PH_REQUIRE(L1 && seg && mp, "prio_sample: null buffer");
  if (prio_one_block((long)N, (long)B)) {
    static_assert(kPsOne >= 2048, "segments of prio_one_block");
    k_prio_one<<<1, kPsThreads, 0, st>>>(L1, (long)N, (long)B, alpha, beta, (unsigned long long)rng, seg, mp);
    PH_LAUNCH_CHECK();
    return PH_OK;
  }
  const size_t tab = (N + 31) & ~(size_t)31;
  double* w = (double*)scratch(kSlotPrio, (N > (size_t)kPsLdsCum ? 2 : 1) * tab * 8);
  if (!w) return PH_ERR_NOMEM;
  k_prio_weights<<<ceil_div(N, 256), 256, 0, st>>>(L1, (long)N, alpha, w);
  if (N <= (size_t)kPsLdsCum)
    k_prio_draws<<<ceil_div(B, kPsDraws), kPsThreads, 0, st>>>(w, (long)N, (long)B, beta, (unsigned long long)rng, seg, mp);
  else
    k_prio_sample<<<1, kPsThreads, 0, st>>>(w, (long)N, (long)B, beta, (unsigned long long)rng, w + tab, seg, mp);
  PH_LAUNCH_CHECK();
  return PH_OK;
}

int mb_gather(const ph_replay_cols& c, const int* seg, const double* mp, size_t B, void* out, double* stats,
              hipStream_t st) {
  const long n = (long)(B * c.T);
  if (n == 0) return PH_OK;
  const int K = c.K ? (int)c.K : 1;
  const bool tiles = sm_tiles(c);
  const unsigned ne = ceil_div((size_t)n, kGaBlock);
  const unsigned nb = tiles ? ceil_div(B, kSm) * ceil_div(c.T, kSt) : ne;
  double* part = (double*)scratch(kSlotReplayPart, (size_t)nb * 3 * 8 + 64);
  if (!part) return PH_ERR_NOMEM;
  if (!stats) {
    stats = (double*)scratch(kSlotReplayStats, 64);
    if (!stats) return PH_ERR_NOMEM;
  }
  const long N = (long)c.N;
  const int T = (int)c.T;
  const bool fold = gather_folds(nb);
#define PH_GATHER_ARGS(R)                                                                                          \
  (const R*)c.adv, (const R*)c.value, (const R*)c.act, (const R*)c.logp, (const R*)c.term, N, T, K, seg, (long)B, \
      (R*)out, part
#define PH_GATHER(R)                                                                                                \
  do {                                                                                                              \
    if (tiles) k_mb_gather_sm<R><<<nb, kGaThreads, 0, st>>>(PH_GATHER_ARGS(R));                                     \
    else if (c.time_major) k_mb_gather<R, true><<<nb, kGaThreads, 0, st>>>(PH_GATHER_ARGS(R));                      \
    else k_mb_gather<R, false><<<nb, kGaThreads, 0, st>>>(PH_GATHER_ARGS(R));                                       \
    R* a = (R*)out + (long)K * n;                                                                                   \
    if (fold) {                                                                                                     \
      k_mb_normalize<R, true><<<ne, kGaThreads, 0, st>>>(a, (long)B, n, mp, part, nb, stats);                       \
    } else {                                                                                                        \
      k_mb_stats<<<1, kGaThreads, 0, st>>>(part, nb, stats);                                                        \
      k_mb_normalize<R, false><<<ne, kGaThreads, 0, st>>>(a, (long)B, n, mp, part, nb, stats);                      \
    }                                                                                                               \
  } while (0)
  if (c.dtype == PH_F64) PH_GATHER(double);
  else PH_GATHER(float);
#undef PH_GATHER
#undef PH_GATHER_ARGS
  PH_LAUNCH_CHECK();
  return PH_OK;
}

int mb_iterate(const ph_replay_cols& c, const int* seg, size_t B, const float* newlp, const float* newval,
               hipStream_t st) {
  if (B == 0) return PH_OK;
  if (iterate_tiled(c.time_major, (long)B, (long)c.T)) {
    const unsigned g = ceil_div(B, kSm) * ceil_div(c.T, kSt);
    if (c.dtype == PH_F64)
      k_mb_iterate_sm<double><<<g, 256, 0, st>>>((double*)c.value, (double*)c.ratio, (const double*)c.logp, newlp,
                                                 newval, seg, (long)B, (long)c.N, (int)c.T);
    else
      k_mb_iterate_sm<float><<<g, 256, 0, st>>>((float*)c.value, (float*)c.ratio, (const float*)c.logp, newlp, newval,
                                                seg, (long)B, (long)c.N, (int)c.T);
    PH_LAUNCH_CHECK();
    return PH_OK;
  }
  int* lw = (int*)scratch_zeroed(kSlotReplayLastw, c.N * 4, st);
  if (!lw) return PH_ERR_NOMEM;
  const long N = (long)c.N;
  const int T = (int)c.T;
  k_mb_lastw<<<ceil_div(B, 256), 256, 0, st>>>(seg, (long)B, N, lw);
  const unsigned g = ceil_div(B, 4);
  if (c.dtype == PH_F64) {
    if (c.time_major)
      k_mb_iterate<double, true><<<g, 256, 0, st>>>((double*)c.value, (double*)c.ratio, (const double*)c.logp,
                                                     newlp, newval, seg, (long)B, N, T, lw);
    else
      k_mb_iterate<double, false><<<g, 256, 0, st>>>((double*)c.value, (double*)c.ratio,
                                                      (const double*)c.logp, newlp, newval, seg, (long)B, N,
                                                      T, lw);
  } else {
    if (c.time_major)
      k_mb_iterate<float, true><<<g, 256, 0, st>>>((float*)c.value, (float*)c.ratio, (const float*)c.logp,
                                                    newlp, newval, seg, (long)B, N, T, lw);
    else
      k_mb_iterate<float, false><<<g, 256, 0, st>>>((float*)c.value, (float*)c.ratio, (const float*)c.logp,
                                                     newlp, newval, seg, (long)B, N, T, lw);
  }
  PH_LAUNCH_CHECK();
  return PH_OK;
}

}  // namespace ph

using namespace ph;

extern "C" int ph_seg_l1(const ph_replay_cols* c, double* L1, void* stream) {
  PH_TRY(check_cols(c, "ph_seg_l1"));
  PH_REQUIRE(c->adv && L1, "ph_seg_l1: null buffer");
  return seg_l1(*c, L1, (hipStream_t)stream);
}

extern "C" int ph_prio_sample(const double* L1, size_t N, size_t Bmb, double alpha, double beta, uint64_t rng,
                              int* seg, double* mbprio, void* stream) {
  return prio_sample(L1, N, Bmb, alpha, beta, rng, seg, mbprio, (hipStream_t)stream);
}

extern "C" int ph_mb_gather(const ph_replay_cols* c, const int* seg, const double* mbprio, size_t Bmb, void* out,
                            double* stats, void* stream) {
  PH_TRY(check_cols(c, "ph_mb_gather"));
  PH_REQUIRE(c->K <= 256, "ph_mb_gather: K=%zu action components", c->K);
  PH_REQUIRE(Bmb <= 0x7fffffffUL && Bmb * c->T <= ((size_t)1 << 40), "ph_mb_gather: Bmb=%zu too large", Bmb);
  if (Bmb == 0) return PH_OK;
  PH_REQUIRE(c->adv && c->value && c->act && c->logp && c->term && seg && out,
             "ph_mb_gather: null buffer");
  return mb_gather(*c, seg, mbprio, Bmb, out, stats, (hipStream_t)stream);
}

extern "C" int ph_mb_iterate(const ph_replay_cols* c, const int* seg, size_t Bmb, const float* newlp,
                             const float* newval, void* stream) {
  PH_TRY(check_cols(c, "ph_mb_iterate"));
  PH_REQUIRE(Bmb <= 0x7fffffffUL, "ph_mb_iterate: Bmb=%zu too large", Bmb);
  if (Bmb == 0) return PH_OK;
  PH_REQUIRE(c->value && c->ratio && c->logp && seg && newlp && newval, "ph_mb_iterate: null buffer");
  return mb_iterate(*c, seg, Bmb, newlp, newval, (hipStream_t)stream);
}
