// Newton-Schulz orthogonalisation of a batch of fp32 matrices on fp32 MFMA (ph_math PH_MATH_F32).
//
// Per step, with the matrices in wide form (m = min(rows, cols) rows, w = max columns):
//   P1  A  = X X^T            lower-triangle tiles, mirrored (A is symmetric to the bit)
//   P2  B  = b A + c A A^T    lower-triangle tiles, mirrored
//   P3  X' = a X + B X        all tiles
// One launch per phase runs the tiles of every matrix of the batch, so a policy's matrices cost the
// launches of one: 2 + 3 per step, against three GEMM calls per step and matrix (with padded operand
// copies for extents off the vector alignment) plus four more each. What bounds these sizes is the chain of
// dependent launches and, inside one, the serial MFMA chain over k: a 32x32 tile per block, whose four
// wavefronts take every fourth 16-wide k chunk of the whole tile, makes that chain four times shorter than
// a quadrant per wavefront, reads each operand element once per block (no LDS staging: both operands are
// k-contiguous, P3's second operand being a transposed copy that the phase writing X also stores), and gives
// a 768x768 matrix 576 tiles where 64x64 ones would leave half the CUs idle. The buffers are zero-padded
// to 32, so no phase guards its loads; leading dimensions are odd multiples of 128 bytes, so that the 16
// rows of a fragment load fall on different L2 channels.
// 5 steps, GEMM chain -> these launches: 96x288 155 -> 85 us, 200x129 394 -> 90, 512x512 469 -> 145, 1536x512
// 419 -> 227, 768x768 404 -> 293; four matrices of a small policy (288x96, 96x40, 5x96, 1x96) 270 -> 86.
#include "common.hpp"
#include "kernels.hpp"
#include "routes.hpp"

namespace ph {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int kTl = 32;          // tile edge
constexpr int kThr = 256;        // four wavefronts, each a quarter of the k chunks
constexpr int kTp = kTl + 4;     // LDS pitch: 16-byte rows, conflict-free accumulator stores
constexpr int kSqChunk = 4096;   // elements per sum-of-squares partial

struct Mat {
  float* x;   // caller's matrix, rows x cols, in place
  float* ws;  // scratch (layout below)
  int rows, cols;
};
struct Launch {
  Mat mat[kNsMaxMats];
  int csq[kNsMaxMats + 1];  // matrix k owns sum-of-squares chunks [csq[k], csq[k + 1])
  int ctri[kNsMaxMats + 1];  // ... lower-triangle tiles
  int call[kNsMaxMats + 1];  // ... tiles of the wide matrix
  int n;
};

struct Geo {
  int m, w, tm, tw, lm, lw;  // extents, tiles, leading dimensions of m- and w-long rows
  bool tall;
  int nsq;
  float *x[2], *xt[2], *a, *b, *part;
};

__host__ __device__ inline int lead(int tiles) { return (tiles | 1) * kTl; }

__host__ __device__ inline size_t layout(const Mat& s, Geo& g) {
  g.tall = s.rows > s.cols;
  g.m = g.tall ? s.cols : s.rows;
  g.w = g.tall ? s.rows : s.cols;
  g.tm = (g.m + kTl - 1) / kTl;
  g.tw = (g.w + kTl - 1) / kTl;
  g.lm = lead(g.tm);
  g.lw = lead(g.tw);
  g.nsq = (int)(((long)s.rows * s.cols + kSqChunk - 1) / kSqChunk);
  const size_t nx = (size_t)g.tm * kTl * g.lw, nt = (size_t)g.tw * kTl * g.lm, nm = (size_t)g.tm * kTl * g.lm;
  float* p = s.ws;
  for (int i = 0; i < 2; i++) {
    g.x[i] = p;
    g.xt[i] = p + nx;
    p += nx + nt;
  }
  g.a = p;
  g.b = p + nm;
  g.part = p + 2 * nm;
  return 2 * (nx + nt) + 2 * nm + (((size_t)g.nsq + 31) & ~(size_t)31);
}

// The matrix that owns item i of a numbering (uniform over the block).
__device__ inline int owner(const int* cum, int n, int i) {
  int k = 0;
  while (k + 1 < n && i >= cum[k + 1]) k++;
  return k;
}

__device__ inline float block_sum(float v, float* sh) {
  sh[threadIdx.x] = v;
  __syncthreads();
  for (int s = kThr / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
    __syncthreads();
  }
  return sh[0];
}

__global__ void __launch_bounds__(kThr) k_nsf_sumsq(Launch L) {
  __shared__ float sh[kThr];
  const int k = owner(L.csq, L.n, blockIdx.x), c = blockIdx.x - L.csq[k];
  Geo g;
  layout(L.mat[k], g);
  const long n = (long)L.mat[k].rows * L.mat[k].cols, lo = (long)c * kSqChunk;
  const float* x = L.mat[k].x;
  float v[kSqChunk / kThr];
#pragma unroll
  for (int i = 0; i < kSqChunk / kThr; i++) {
    const long e = lo + i * kThr + threadIdx.x;
    v[i] = e < n ? x[e] : 0.f;
  }
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < kSqChunk / kThr; i++) s += v[i] * v[i];
  s = block_sum(s, sh);
  if (threadIdx.x == 0) g.part[c] = s;
}

// X = x / (||x||_F + eps) in wide form and transposed, zero past the extents. Tiles are walked in the
// source's own orientation: its rows are the wide rows, or (tall) the transposed ones.
__global__ void __launch_bounds__(kThr) k_nsf_load(Launch L, float eps) {
  __shared__ float sh[kThr];
  __shared__ float tl[kTl][kTl + 1];
  const int k = owner(L.call, L.n, blockIdx.x), t = blockIdx.x - L.call[k];
  const Mat s = L.mat[k];
  Geo g;
  layout(s, g);
  const int ti = t % g.tm, tj = t / g.tm;
  const int r0 = (g.tall ? tj : ti) * kTl, c0 = (g.tall ? ti : tj) * kTl;
  const int c = threadIdx.x & 31, r = threadIdx.x >> 5;
  float v[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int rr = r0 + r + 8 * i, cc = c0 + c;
    v[i] = rr < s.rows && cc < s.cols ? s.x[(long)rr * s.cols + cc] : 0.f;
  }
  float q = 0.f;
  for (int i = threadIdx.x; i < g.nsq; i += kThr) q += g.part[i];
  const float inv = 1.f / (sqrtf(block_sum(q, sh)) + eps);
  float* nat = g.tall ? g.xt[0] : g.x[0];
  float* tra = g.tall ? g.x[0] : g.xt[0];
  const int ln = g.tall ? g.lm : g.lw, lt = g.tall ? g.lw : g.lm;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const float y = inv * v[i];
    nat[(long)(r0 + r + 8 * i) * ln + c0 + c] = y;
    tl[r + 8 * i][c] = y;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; i++) tra[(long)(c0 + r + 8 * i) * lt + r0 + c] = tl[c][r + 8 * i];
}

// One 32x32 tile of a phase. Fragments come straight from memory: lane l of a wavefront loads 16 bytes of
// row l % 16 at k offset 4 (l / 16) of a 16-wide chunk, and MFMA e (of four) takes element e, i.e. the k
// values e, 4 + e, 8 + e and 12 + e of both operands. Two chunks are multiplied while the next two load.
template <int P>
__global__ void __launch_bounds__(kThr) k_nsf_tile(Launch L, int step, int last, float ca, float cb, float cc) {
  __shared__ float red[4][kTl][kTp];
  const int* cum = P == 3 ? L.call : L.ctri;
  const int k = owner(cum, L.n, blockIdx.x), t = blockIdx.x - cum[k];
  const Mat s = L.mat[k];
  Geo g;
  layout(s, g);
  int ti, tj;
  if (P == 3) {
    ti = t % g.tm;
    tj = t / g.tm;
  } else {
    ti = (int)((sqrtf(8.f * (float)t + 1.f) - 1.f) * 0.5f);
    while (ti * (ti + 1) / 2 > t) ti--;
    while ((ti + 1) * (ti + 2) / 2 <= t) ti++;
    tj = t - ti * (ti + 1) / 2;
  }
  const int in = step & 1;
  const float* o1 = P == 1 ? g.x[in] : P == 2 ? g.a : g.b;
  const float* o2 = P == 1 ? g.x[in] : P == 2 ? g.a : g.xt[in];
  const int ld = P == 1 ? g.lw : g.lm;
  const int nc = 2 * (P == 1 ? g.tw : g.tm);
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int fr = lane & 15, fg = lane >> 4;
  const float* pa = o1 + (long)(ti * kTl + fr) * ld + 4 * fg;
  const float* pb = o2 + (long)(tj * kTl + fr) * ld + 4 * fg;
  f4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) acc[i][j] = (f4){0.f, 0.f, 0.f, 0.f};
  f4 cur[2][4], nxt[2][4];
  auto load = [&](int c, f4 (&f)[4]) {
    if (c < nc) {
      f[0] = *(const f4*)(pa + 16 * c);
      f[1] = *(const f4*)(pa + 16 * c + (long)16 * ld);
      f[2] = *(const f4*)(pb + 16 * c);
      f[3] = *(const f4*)(pb + 16 * c + (long)16 * ld);
    } else {
#pragma unroll
      for (int i = 0; i < 4; i++) f[i] = (f4){0.f, 0.f, 0.f, 0.f};
    }
  };
  auto mul = [&](const f4 (&f)[4]) {
#pragma unroll
    for (int e = 0; e < 4; e++)
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(f[i][e], f[2 + j][e], acc[i][j], 0, 0, 0);
  };
  load(wv, cur[0]);
  load(wv + 4, cur[1]);
  for (int c = wv; c < nc; c += 8) {
    load(c + 8, nxt[0]);
    load(c + 12, nxt[1]);
    mul(cur[0]);
    if (c + 4 < nc) mul(cur[1]);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      cur[0][i] = nxt[0][i];
      cur[1][i] = nxt[1][i];
    }
  }
  // accumulator element e of lane (fr, fg): row 4 fg + e, column fr
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int e = 0; e < 4; e++) red[wv][16 * i + 4 * fg + e][16 * j + fr] = acc[i][j][e];
  __syncthreads();
  const int r = threadIdx.x >> 3, c4 = 4 * (threadIdx.x & 7);
  const f4 s01 = *(const f4*)&red[0][r][c4] + *(const f4*)&red[1][r][c4];
  const f4 s23 = *(const f4*)&red[2][r][c4] + *(const f4*)&red[3][r][c4];
  f4 v = s01 + s23;
  const int row = ti * kTl + r, col = tj * kTl + c4;
  if (P == 2) v = cb * *(const f4*)(g.a + (long)row * g.lm + col) + cc * v;
  if (P == 3) v = ca * *(const f4*)(g.x[in] + (long)row * g.lw + col) + v;
  const bool flip = P == 3 ? (!last || g.tall) : ti != tj;
  if (flip) {  // the tile transposed: the mirror of a symmetric product, or X'^T
    __syncthreads();
    *(f4*)&red[0][r][c4] = v;
    __syncthreads();
  }
  f4 vt = {0.f, 0.f, 0.f, 0.f};
  if (flip)
#pragma unroll
    for (int e = 0; e < 4; e++) vt[e] = red[0][c4 + e][r];
  const int trow = tj * kTl + r, tcol = ti * kTl + c4;
  if (P == 3 && last) {
    const f4 y = g.tall ? vt : v;
    const int yr = g.tall ? trow : row, yc = g.tall ? tcol : col;
    if (yr < s.rows)
#pragma unroll
      for (int e = 0; e < 4; e++)
        if (yc + e < s.cols) s.x[(long)yr * s.cols + yc + e] = y[e];
  } else {
    float* d = P == 1 ? g.a : P == 2 ? g.b : g.x[in ^ 1];
    *(f4*)(d + (long)row * (P == 3 ? g.lw : g.lm) + col) = v;
    if (flip) *(f4*)((P == 3 ? g.xt[in ^ 1] : d) + (long)trow * g.lm + tcol) = vt;
  }
}

}  // namespace

int ns_f32_batch(float* const* X, const int* rows, const int* cols, int n, const float* coeffs, int nsteps, float eps,
                 int ws_slot, hipStream_t st) {
  if (nsteps < 1) {
    set_error("newton_schulz (fp32): no steps");
    return PH_ERR_UNSUPPORTED;
  }
  for (int i = 0; i < n;) {
    Launch L{};
    size_t off[kNsMaxMats], words = 0;
    for (; i < n && L.n < kNsMaxMats; i++) {
      if ((long)rows[i] * cols[i] == 0) continue;
      if (!ns_f32_fits(rows[i], cols[i])) {
        set_error("newton_schulz (fp32): %d x %d does not fit the batched launches", rows[i], cols[i]);
        return PH_ERR_UNSUPPORTED;
      }
      const int k = L.n++;
      L.mat[k] = Mat{X[i], nullptr, rows[i], cols[i]};
      Geo g;
      off[k] = words;
      words += layout(L.mat[k], g);
      L.csq[k + 1] = L.csq[k] + g.nsq;
      L.ctri[k + 1] = L.ctri[k] + g.tm * (g.tm + 1) / 2;
      L.call[k + 1] = L.call[k] + g.tm * g.tw;
    }
    if (L.n == 0) continue;
    float* ws = (float*)scratch(ws_slot, words * 4);
    if (!ws) return PH_ERR_NOMEM;
    for (int k = 0; k < L.n; k++) L.mat[k].ws = ws + off[k];
    k_nsf_sumsq<<<L.csq[L.n], kThr, 0, st>>>(L);
    k_nsf_load<<<L.call[L.n], kThr, 0, st>>>(L, eps);
    for (int s = 0; s < nsteps; s++) {
      const float a = coeffs[3 * s], b = coeffs[3 * s + 1], c = coeffs[3 * s + 2];
      k_nsf_tile<1><<<L.ctri[L.n], kThr, 0, st>>>(L, s, 0, a, b, c);
      k_nsf_tile<2><<<L.ctri[L.n], kThr, 0, st>>>(L, s, 0, a, b, c);
      k_nsf_tile<3><<<L.call[L.n], kThr, 0, st>>>(L, s, s + 1 == nsteps, a, b, c);
    }
    PH_LAUNCH_CHECK();
  }
  return PH_OK;
}

}  // namespace ph
