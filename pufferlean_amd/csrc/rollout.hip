// Rollout policy forward and categorical sampler: what produces the behaviour log-prob and value
// columns the update consumes.
//
//   ph_sample_actions       categorical draw per row of logits      (k_sample / k_sample_f32,
//                                                                     puffercuda.cu:1429-1460; CPU twin
//                                                                     pufferffi.c:896-918)
//   ph_mingru_rollout_step  one timestep of the MinGRU policy       (lean_cuda_mingru_step,
//                           over N envs, state carried in place      puffercuda.cu:2190-2265)
//
// The step runs the encoder (bias fused) on the MFMA GEMM, then one kernel per layer that forms a unit's hid,
// gate and proj products in one wavefront's accumulators and applies the cell to them in registers, and one
// kernel for the head (action logits and the value, bias fused, written straight into the [N][A+1]
// output). Hidden sizes that are no multiple of 8, and the large ones rollout_form leaves, run the products on the
// GEMM, a cell kernel and a padded head instead.
// Its launches are plain stream work, so a caller can capture a whole horizon in one HIP graph.
#include <cmath>
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"
#include "routes.hpp"

// The sampler's formulas execute in the order written (no fused multiply-add), as in the CPU twin.
#pragma clang fp contract(off)

namespace ph {
namespace {

constexpr int HP = 32;  // padded head rows: A logits, the value, zeros

__device__ __forceinline__ unsigned long long sm64_mix(unsigned long long z) {
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
  return z ^ (z >> 31);
}
__device__ __forceinline__ float ex(float x) { return expf(x); }
__device__ __forceinline__ double ex(double x) { return exp(x); }
__device__ __forceinline__ float lg(float x) { return logf(x); }
__device__ __forceinline__ double lg(double x) { return log(x); }

// Row n (stride ldy): m = max of the A logits, z = sum exp(l - m); the draw u is the top 53 bits of
// the splitmix64 word of rng + (n+1)*GOLD over 2^53; the action is the first k whose running sum of
// exp(l_k - m)/z exceeds u (A-1 if none); logp = log(exp(l_a - m)/z); the value is column A. R is the
// logit type (the running sum and logp are in R; u is always f64, as in the reference's f32 form).
// Bound by latency (one row per lane, 17 columns at a rollout): with AMAX > 0 (A <= AMAX) the row is loaded
// into registers at once and each exponential is formed once, in blocks of one wavefront so that 4096 rows
// spread over 64 CUs; AMAX = 0 reads the row from memory in each pass (sample_registers chooses). The same
// expressions in the same order: 4096 rows of 16, 8.4 -> 3.8 us.
template <typename R, bool OUT3, int AMAX>
__global__ void __launch_bounds__(256) k_sample_cat(const R* __restrict__ Y, long ldy, long N, int A,
                                                    int has_value, unsigned long long rng, int* __restrict__ act,
                                                    R* __restrict__ logp, R* __restrict__ val,
                                                    double* __restrict__ out3) {
  const long n = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= N) return;
  const R* row = Y + n * ldy;
  const R v = has_value ? row[A] : R(0);
  R x[AMAX ? AMAX : 1];
  if constexpr (AMAX > 0) {
#pragma unroll
    for (int k = 0; k < AMAX; k++) x[k] = row[k < A ? k : A - 1];
  }
  R m = row[0], z = 0;
  if constexpr (AMAX > 0) {
#pragma unroll
    for (int k = 1; k < AMAX; k++)
      if (k < A && x[k] > m) m = x[k];
#pragma unroll
    for (int k = 0; k < AMAX; k++) {
      x[k] = ex(x[k] - m);
      if (k < A) z += x[k];
    }
  } else {
    for (int k = 1; k < A; k++)
      if (row[k] > m) m = row[k];
    for (int k = 0; k < A; k++) z += ex(row[k] - m);
  }
  const unsigned long long w = sm64_mix(rng + (unsigned long long)(n + 1) * 0x9E3779B97F4A7C15ULL);
  const double u = (double)(w >> 11) / 9007199254740992.0;
  R acc = 0;
  int a = A - 1;
  R pa = 0;  // the drawn action's probability
  if constexpr (AMAX > 0) {
    bool open = true;
#pragma unroll
    for (int k = 0; k < AMAX; k++)
      if (k < A && open) {
        pa = x[k] / z;
        acc += pa;
        if (u < (double)acc) {
          a = k;
          open = false;
        }
      }
  } else {
    for (int k = 0; k < A; k++) {
      pa = ex(row[k] - m) / z;
      acc += pa;
      if (u < (double)acc) {
        a = k;
        break;
      }
    }
  }
  const R lp = lg(pa);
  if (act) act[n] = a;
  if (logp) logp[n] = lp;
  if (val) val[n] = v;
  if constexpr (OUT3) {
    out3[n] = (double)a;
    out3[N + n] = (double)lp;
    out3[2 * N + n] = (double)v;
  }
}

// The MinGRU cell of layer l for one step (the reference's k_mingru_gate, puffercuda.cu:1949-1959):
// cmb [N][3H] = hid | gate | proj of this layer's product, xin [N][H] the layer input, state [N][L][H].
//   o = (1 - sigmoid(gate)) * prev + sigmoid(gate) * gact(hid),  gact(x) = x >= 0 ? x + 1/2 : sigmoid(x)
//   xout = sigmoid(proj) * o + (1 - sigmoid(proj)) * xin,  state <- o
__device__ __forceinline__ float sig_ieee(float x) { return 1.0f / (1.0f + expf(-x)); }
__global__ void __launch_bounds__(256) k_rollout_cell(const float* __restrict__ cmb, const float* __restrict__ xin,
                                                      float* __restrict__ state, float* __restrict__ xout, long N,
                                                      int L, int H, int l) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= N * H) return;
  const long n = idx / H;
  const int j = (int)(idx - n * H);
  const float* y = cmb + n * 3 * H;
  const float hid = y[j], gate = y[H + j], proj = y[2 * H + j];
  const float zg = sig_ieee(gate), g = hid >= 0.f ? hid + 0.5f : sig_ieee(hid), hg = sig_ieee(proj);
  float* s = state + (n * L + l) * H + j;
  const float o = (1.0f - zg) * *s + zg * g;
  xout[idx] = hg * o + (1.0f - hg) * xin[idx];
  *s = o;
}

// ---- layer and head on MFMA with the cell fused (H a multiple of 8) -------------------------------------
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));  // the value row's offset may be odd

__device__ __forceinline__ u32x4 cvt8(const f32x4& a, const f32x4& b) {
  return {bf16x2_rne(a[0], a[1]), bf16x2_rne(a[2], a[3]), bf16x2_rne(b[0], b[1]), bf16x2_rne(b[2], b[3])};
}
__device__ __forceinline__ void mma_bf(floatx16& c, const u32x4& a, const u32x4& b) {
  c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0,
                                              0, 0);
}
__device__ __forceinline__ void mma_f32(floatx16& c, const f32x4& a, const f32x4& b) {
#pragma unroll
  for (int q = 0; q < 4; q++) c = __builtin_amdgcn_mfma_f32_32x32x2f32(a[q], b[q], c, 0, 0, 0);
}
__device__ __forceinline__ void lds_sync() {  // orders LDS only: prefetched loads stay in flight
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// One cell (k_rollout_cell's expressions).
__device__ __forceinline__ float cell(float hid, float gate, float proj, float prev, float xin, float& o) {
  const float zg = sig_ieee(gate), g = hid >= 0.f ? hid + 0.5f : sig_ieee(hid), hg = sig_ieee(proj);
  o = (1.0f - zg) * prev + zg * g;
  return hg * o + (1.0f - hg) * xin;
}

// Layer l over tiles of 32 NW rows x 32 units: a wavefront holds the hid, gate and proj products of its 32 rows
// and the 32 units, so the cell runs on its accumulators and the [N][3H] products never reach memory (they were
// 50 MB of a 4096 x 512 step's traffic, and the cell a launch of 10.6 us). X: the layer input in the
// product's type (bf16 copy or fp32), xin the same in fp32 for the cell's skip; the fp32 weights are rounded on
// their way into LDS. Operands into the CUs are what a block moves most of (256 rows x 96 weight rows, one block
// per CU at 4096 x 512); two k chunks in flight in registers, LDS double-buffered. rollout_form chooses NW.
// 4096 rows, H 512: 19.9 + 10.6 us -> about 22 (bf16 products); the whole step 89 -> 59 us, fp32 208 -> 157.
template <bool BF, int NW>
__global__ void __launch_bounds__(64 * NW, 1) k_roll_layer(const void* __restrict__ X, const float* __restrict__ xin,
                                                        const float* __restrict__ W, float* __restrict__ state,
                                                        float* __restrict__ xout, uint16_t* __restrict__ xoutb, long N,
                                                        int L, int H, int l) {
  constexpr int NT = 64 * NW, R = 32 * NW;
  constexpr int BK = BF ? 64 : 32;         // k per chunk: 8 pieces per row either way
  constexpr int EL = BF ? 8 : 4;           // k per piece
  constexpr int ES = BF ? 2 : 4;
  constexpr int PB = (BK + EL) * ES;       // LDS row pitch in bytes: 144, conflict-free 16-byte reads
  constexpr int CA = R * 8 / NT, CB = (96 * 8 + NT - 1) / NT;
  static_assert(2 * (R + 96) * PB <= 160 * 1024, "LDS budget");
  __shared__ __align__(16) uint8_t sm[2][(R + 96) * PB];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lr = lane & 31, half = lane >> 5;
  const long m0 = (long)blockIdx.x * R;
  const int j0 = blockIdx.y * 32;
  struct Set {
    u32x4 a[CA];
    f32x4 b[CB][BF ? 2 : 1];
  } rg[2];
  const int nk = (H + BK - 1) / BK;
  auto gload = [&](Set& s, int c) {
#pragma unroll
    for (int i = 0; i < CA; i++) {
      const int id = tid + i * NT, k = min(c * BK + (id & 7) * EL, H - EL);
      const long n = m0 + (id >> 3) < N ? m0 + (id >> 3) : N - 1;
      s.a[i] = *reinterpret_cast<const u32x4*>(reinterpret_cast<const uint8_t*>(X) + (n * H + k) * ES);
    }
#pragma unroll
    for (int i = 0; i < CB; i++) {
      const int id = min(tid + i * NT, 96 * 8 - 1), q = id >> 3, k = min(c * BK + (id & 7) * EL, H - EL);
      const float* p = W + ((long)(q >> 5) * H + min(j0 + (q & 31), H - 1)) * H + k;
#pragma unroll
      for (int h = 0; h < (BF ? 2 : 1); h++) s.b[i][h] = reinterpret_cast<const f32x4*>(p)[h];
    }
  };
  // a piece past the end of k is stored as zero (the loads re-read the row's last piece)
  auto sstore = [&](const Set& s, int c, int buf) {
#pragma unroll
    for (int i = 0; i < CA; i++) {
      const int id = tid + i * NT;
      const bool in = c * BK + (id & 7) * EL < H;
      *reinterpret_cast<u32x4*>(&sm[buf][(id >> 3) * PB + (id & 7) * 16]) = in ? s.a[i] : u32x4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int i = 0; i < CB; i++) {
      const int id = tid + i * NT;
      if (id < 96 * 8) {
        u32x4 v;
        if constexpr (BF) v = cvt8(s.b[i][0], s.b[i][1]);
        else v = __builtin_bit_cast(u32x4, s.b[i][0]);
        const bool in = c * BK + (id & 7) * EL < H;
        *reinterpret_cast<u32x4*>(&sm[buf][(R + (id >> 3)) * PB + (id & 7) * 16]) = in ? v : u32x4{0u, 0u, 0u, 0u};
      }
    }
  };
  floatx16 acc[3];
#pragma unroll
  for (int t = 0; t < 3; t++)
#pragma unroll
    for (int r = 0; r < 16; r++) acc[t][r] = 0.f;
  auto compute = [&](int buf) {
    const uint8_t* pa = &sm[buf][(wave * 32 + lr) * PB + half * 16];
    const uint8_t* pb = &sm[buf][(R + lr) * PB + half * 16];
#pragma unroll
    for (int q = 0; q < 4; q++) {  // two pieces of k: the lower half-wavefront's, the upper's
      if constexpr (BF) {
        const u32x4 a = *reinterpret_cast<const u32x4*>(pa + q * 32);
#pragma unroll
        for (int t = 0; t < 3; t++) mma_bf(acc[t], a, *reinterpret_cast<const u32x4*>(pb + t * 32 * PB + q * 32));
      } else {
        const f32x4 a = *reinterpret_cast<const f32x4*>(pa + q * 32);
#pragma unroll
        for (int t = 0; t < 3; t++) mma_f32(acc[t], a, *reinterpret_cast<const f32x4*>(pb + t * 32 * PB + q * 32));
      }
    }
  };
  gload(rg[0], 0);
  gload(rg[1], 1);
  // the cell's operands, in flight through the k loop (32-bit offsets from the tile's first row)
  const int j = j0 + lr;
  const float* const sp = state + (m0 * L + l) * H + min(j, H - 1);
  const float* const xp = xin + m0 * H + min(j, H - 1);
  const int rmax = (int)min((long)R, N - m0) - 1, rb = wave * 32 + 4 * half;
  float prev[16], xi[16];
#pragma unroll
  for (int e = 0; e < 16; e++) {
    const int r = min(rb + 8 * (e >> 2) + (e & 3), rmax);
    prev[e] = sp[r * L * H];
    xi[e] = xp[r * H];
  }
  sstore(rg[0], 0, 0);
  lds_sync();
  for (int c = 0; c < nk; c += 2) {
    gload(rg[0], c + 2);
    compute(0);
    sstore(rg[1], c + 1, 1);
    lds_sync();
    if (c + 1 >= nk) break;
    gload(rg[1], c + 3);
    compute(1);
    sstore(rg[0], c + 2, 0);
    lds_sync();
  }
  if (j >= H) return;
#pragma unroll
  for (int e = 0; e < 16; e++) {
    const int r = rb + 8 * (e >> 2) + (e & 3);
    if (r > rmax) continue;
    float o;
    const float h = cell(acc[0][e], acc[1][e], acc[2][e], prev[e], xi[e], o);
    state[(m0 * L + l) * H + j + r * L * H] = o;
    xout[m0 * H + j + r * H] = h;
    if constexpr (BF) xoutb[m0 * H + j + r * H] = bf16_rne(h);
  }
}

// Few rows: 32 rows x 32 units a block, k split over its four wavefronts with fragments loaded straight into
// registers (no LDS round trip, every load of a wavefront in flight at once), the partial sums added in
// wavefront order through LDS. TILES = 3: a layer with the cell; TILES = 1: the head, whose row c is W's
// row c for c < A and the value row Wv for c = A. Bound by launch and load latency.
// 48 rows, H 128, fp32: layer product and cell 6.2 + 2.6 us -> 7.9 us; the head at 4096 rows of 512 (a split-K
// GEMM on a padded copy, 15.5 + 4.3 + 2.5 us) -> 4.8 us.
template <bool BF, int TILES>
__global__ void __launch_bounds__(256) k_roll_reg(const void* __restrict__ X, const float* __restrict__ xin,
                                                  const float* __restrict__ W, const float* __restrict__ Wv,
                                                  const float* __restrict__ bias, const float* __restrict__ biasv,
                                                  float* __restrict__ state, float* __restrict__ out,
                                                  uint16_t* __restrict__ outb, long N, int L, int H, int l, int A) {
  constexpr int KS = BF ? 16 : 8;  // k per step (one fragment per lane)
  constexpr int U = 4;             // steps in flight
  constexpr int ES = BF ? 2 : 4;
  __shared__ float red[4][TILES * 16][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lr = lane & 31, half = lane >> 5;
  const long m0 = (long)blockIdx.x * 32;
  const int j0 = blockIdx.y * 32;
  const long n = min(m0 + lr, N - 1);
  const uint8_t* pa = reinterpret_cast<const uint8_t*>(X) + n * H * ES;
  const float* pb[TILES];
#pragma unroll
  for (int t = 0; t < TILES; t++) {
    if constexpr (TILES == 3) pb[t] = W + ((long)t * H + min(j0 + lr, H - 1)) * H;
    else pb[t] = lr < A ? W + (long)lr * H : Wv;  // columns past A are not stored
  }
  floatx16 acc[TILES];
#pragma unroll
  for (int t = 0; t < TILES; t++)
#pragma unroll
    for (int r = 0; r < 16; r++) acc[t][r] = 0.f;
  const int ns = (H + KS - 1) / KS;
  for (int s0 = wave; s0 < ns; s0 += 4 * U) {
    u32x4 a[U];
    f32x4 b[U][TILES][BF ? 2 : 1];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int k = (s0 + 4 * u) * KS + half * (KS / 2);
      const int kc = min(k, H - KS / 2);
      a[u] = *reinterpret_cast<const u32x4*>(pa + (long)kc * ES);
      if (k >= H) a[u] = u32x4{0u, 0u, 0u, 0u};  // past the end: zero times a valid weight
#pragma unroll
      for (int t = 0; t < TILES; t++)
#pragma unroll
        for (int h = 0; h < (BF ? 2 : 1); h++) {
          b[u][t][h] = reinterpret_cast<const f32x4u*>(pb[t] + kc)[h];
          if (k >= H) b[u][t][h] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int t = 0; t < TILES; t++) {
        if constexpr (BF) mma_bf(acc[t], a[u], cvt8(b[u][t][0], b[u][t][1]));
        else mma_f32(acc[t], __builtin_bit_cast(f32x4, a[u]), b[u][t][0]);
      }
  }
#pragma unroll
  for (int t = 0; t < TILES; t++)
#pragma unroll
    for (int r = 0; r < 16; r++) red[wave][t * 16 + r][lane] = acc[t][r];
  __syncthreads();
  // wavefront w finishes accumulator elements 4w .. 4w + 3 (rows 8w + 4 half + 0..3)
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const long row = m0 + 8 * wave + 4 * half + q;
    float v[TILES];
#pragma unroll
    for (int t = 0; t < TILES; t++) {
      const int e = t * 16 + 4 * wave + q;
      v[t] = ((red[0][e][lane] + red[1][e][lane]) + red[2][e][lane]) + red[3][e][lane];
    }
    if (row >= N) continue;
    if constexpr (TILES == 3) {
      const int j = j0 + lr;
      if (j < H) {
        float* st = state + (row * L + l) * H + j;
        float o;
        const float h = cell(v[0], v[1], v[2], *st, xin[row * H + j], o);
        *st = o;
        out[row * H + j] = h;
        if constexpr (BF) outb[row * H + j] = bf16_rne(h);
      }
    } else if (lr <= A) {
      out[row * (A + 1) + lr] = v[0] + (lr < A ? bias[lr] : biasv[0]);
    }
  }
}

// Padded head [HP][H] (rows: wDec, wVal, zeros) and its bias [HP] from the flat parameters.
__global__ void k_rollout_head(const float* __restrict__ p, int D, int H, int L, int A, float* __restrict__ wh,
                               float* __restrict__ bh) {
  const long offDec = (long)H * D + H + (long)L * 3 * H * H, offBDec = offDec + (long)A * H,
             offVal = offBDec + A, offBVal = offVal + H;
  const long n = (long)HP * H + HP;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    if (i < (long)HP * H) {
      const int row = (int)(i / H), col = (int)(i % H);
      wh[i] = row < A ? p[offDec + (long)row * H + col] : (row == A ? p[offVal + col] : 0.f);
    } else {
      const int k = (int)(i - (long)HP * H);
      bh[k] = k < A ? p[offBDec + k] : (k == A ? p[offBVal] : 0.f);
    }
  }
}

PhGemmDesc nt_f32(int M, int N, int K, const float* A, long lda, const float* B, long ldb, float* C, long ldc,
                  int math) {
  PhGemmDesc d{};
  d.trans_a = 0; d.trans_b = 1; d.M = M; d.N = N; d.K = K;
  d.a_dtype = PH_F32; d.A = A; d.lda = lda; d.b_dtype = PH_F32; d.B = B; d.ldb = ldb;
  d.c_dtype = PH_F32; d.C = C; d.ldc = ldc; d.math = math; d.alpha = 1.f;
  return d;
}

}  // namespace

int sample_actions(int dtype, const void* Y, size_t ldy, size_t N, size_t A, int has_value, uint64_t rng, int* act,
                   void* logp, void* val, double* out3, hipStream_t st) {
  if (N == 0) return PH_OK;
  // rows in registers: 64 rows a block
  auto go = [&](auto zero, auto amax) {
    using R = decltype(zero);
    constexpr int AM = decltype(amax)::value, BT = AM ? 64 : 256;
    const unsigned g = ceil_div(N, BT);
    if (out3)
      k_sample_cat<R, true, AM><<<g, BT, 0, st>>>((const R*)Y, (long)ldy, (long)N, (int)A, has_value, rng, act, (R*)logp,
                                                 (R*)val, out3);
    else
      k_sample_cat<R, false, AM><<<g, BT, 0, st>>>((const R*)Y, (long)ldy, (long)N, (int)A, has_value, rng, act,
                                                  (R*)logp, (R*)val, nullptr);
  };
  auto width = [&](auto zero) {
    switch (sample_registers((long)A)) {
      case 4: go(zero, std::integral_constant<int, 4>{}); break;
      case 8: go(zero, std::integral_constant<int, 8>{}); break;
      case 16: go(zero, std::integral_constant<int, 16>{}); break;
      case 32: go(zero, std::integral_constant<int, 32>{}); break;
      default: go(zero, std::integral_constant<int, 0>{});
    }
  };
  if (dtype == PH_F64) width(0.0);
  else width(0.f);
  PH_LAUNCH_CHECK();
  return PH_OK;
}

template <bool BF>
void launch_layer(RollForm form, const void* X, const float* xin, const float* W, float* state, float* xout,
                  uint16_t* xoutb, long N, int L, int H, int l, hipStream_t st) {
  const unsigned gj = ceil_div(H, 32);
  if (form == kRoll32) {
    k_roll_reg<BF, 3><<<dim3(ceil_div(N, 32), gj), 256, 0, st>>>(X, xin, W, nullptr, nullptr, nullptr, state, xout,
                                                                 xoutb, N, L, H, l, 0);
    return;
  }
  if constexpr (BF)
    if (form == kRoll256) {
      k_roll_layer<BF, 8><<<dim3(ceil_div(N, 256), gj), 512, 0, st>>>(X, xin, W, state, xout, xoutb, N, L, H, l);
      return;
    }
  k_roll_layer<BF, 4><<<dim3(ceil_div(N, 128), gj), 256, 0, st>>>(X, xin, W, state, xout, xoutb, N, L, H, l);
}

template <bool BF>
int rollout_fused(RollForm form, const ph_mingru_dims& d, const float* params, const float* obs, float* state,
                  float* out, hipStream_t st) {
  const long N = d.B;
  const int D = d.D, H = d.H, L = d.L, A = d.A;
  const size_t nx = ((size_t)N * H + 63) & ~(size_t)63;
  float* base = (float*)scratch(kSlotRollout, nx * (BF ? 3 : 2) * 4);
  if (!base) return PH_ERR_NOMEM;
  float* x[2] = {base, base + nx};
  uint16_t* xb[2] = {(uint16_t*)(base + 2 * nx), (uint16_t*)(base + 2 * nx) + nx};
  PhGemmDesc g = nt_f32((int)N, H, D, obs, D, params, D, x[0], H, BF ? PH_MATH_BF16 : PH_MATH_F32);
  g.epi = PH_EPI_BIAS;
  g.bias = params + (long)H * D;
  if (BF) {
    g.C2 = xb[0];
    g.ldc2 = H;
  }
  PH_TRY(gemm(g, st));
  const float* wl = params + (long)H * D + H;
  auto in = [&](int i) { return BF ? (const void*)xb[i] : (const void*)x[i]; };
  for (int l = 0; l < L; l++) {
    launch_layer<BF>(form, in(l & 1), x[l & 1], wl + (long)l * 3 * H * H, state, x[(l + 1) & 1], xb[(l + 1) & 1], N, L, H, l,
                     st);
    PH_LAUNCH_CHECK();
  }
  const float *wd = wl + (long)L * 3 * H * H, *bd = wd + (long)A * H, *wv = bd + A, *bv = wv + H;
  k_roll_reg<BF, 1><<<ceil_div(N, 32), 256, 0, st>>>(in(L & 1), nullptr, wd, wv, bd, bv, nullptr, out, nullptr, N, L, H,
                                                     0, A);
  PH_LAUNCH_CHECK();
  return PH_OK;
}

int mingru_rollout_step(const ph_mingru_dims& d, const float* params, const float* obs, float* state, float* out,
                        hipStream_t st) {
  const long N = d.B;
  const int D = d.D, H = d.H, L = d.L, A = d.A;
  const int math = d.precision ? PH_MATH_F32 : PH_MATH_BF16;
  // the fused kernels read weight rows and layer inputs in 16- and 32-byte pieces along k: whole pieces need
  // H a multiple of 8, and 16-byte alignment of the layers' rows (they start at H D + H floats, then a
  // multiple of 8; the head's value row may sit at any offset and is read with 4-byte alignment).
  const RollForm form =
      H % 8 == 0 && ((uintptr_t)params & 15) == 0 ? rollout_form(!d.precision, N, H) : kRollChain;
  if (form != kRollChain)
    return d.precision ? rollout_fused<false>(form, d, params, obs, state, out, st)
                       : rollout_fused<true>(form, d, params, obs, state, out, st);
  const size_t nx = (size_t)N * H;
  float* base = (float*)scratch(kSlotRollout, (2 * nx + (size_t)N * 3 * H + (size_t)HP * H + HP) * 4);
  if (!base) return PH_ERR_NOMEM;
  float* x[2] = {base, base + nx};
  float* cmb = base + 2 * nx;
  float* wh = cmb + (size_t)N * 3 * H;
  float* bh = wh + (size_t)HP * H;
  k_rollout_head<<<ceil_div((size_t)HP * H + HP, 256), 256, 0, st>>>(params, D, H, L, A, wh, bh);
  PH_LAUNCH_CHECK();
  PhGemmDesc g = nt_f32((int)N, H, D, obs, D, params, D, x[0], H, math);
  g.epi = PH_EPI_BIAS;
  g.bias = params + (long)H * D;
  PH_TRY(gemm(g, st));
  const float* wl = params + (long)H * D + H;
  for (int l = 0; l < L; l++) {
    g = nt_f32((int)N, 3 * H, H, x[l & 1], H, wl + (long)l * 3 * H * H, H, cmb, 3 * H, math);
    PH_TRY(gemm(g, st));
    k_rollout_cell<<<ceil_div(nx, 256), 256, 0, st>>>(cmb, x[l & 1], state, x[(l + 1) & 1], N, L, H, l);
    PH_LAUNCH_CHECK();
  }
  g = nt_f32((int)N, A + 1, H, x[L & 1], H, wh, H, out, A + 1, math);
  g.epi = PH_EPI_BIAS;
  g.bias = bh;
  return gemm(g, st);
}

}  // namespace ph

using namespace ph;

extern "C" int ph_sample_actions(int dtype, const void* Y, size_t ldy, size_t N, size_t A, int has_value,
                                 uint64_t rng, int* act, void* logp, void* value, void* stream) {
  PH_REQUIRE(dtype == PH_F32 || dtype == PH_F64, "ph_sample_actions: dtype must be PH_F32 or PH_F64");
  PH_REQUIRE(A >= 1 && ldy >= A + (has_value ? 1 : 0), "ph_sample_actions: A=%zu ldy=%zu", A, ldy);
  PH_REQUIRE(N <= 0x7fffffffUL, "ph_sample_actions: N=%zu", N);
  if (N == 0) return PH_OK;
  PH_REQUIRE(Y, "ph_sample_actions: null logits");
  return sample_actions(dtype, Y, ldy, N, A, has_value, rng, act, logp, value, nullptr, (hipStream_t)stream);
}

extern "C" int ph_mingru_rollout_step(const ph_mingru_dims* d, const float* params, const float* obs, float* state,
                                      float* out, void* stream) {
  PH_REQUIRE(d && params && obs && state && out, "ph_mingru_rollout_step: null argument");
  PH_REQUIRE(d->B > 0 && d->D > 0 && d->H > 0 && d->L > 0 && d->A > 0 && d->A + 1 <= HP,
             "ph_mingru_rollout_step: envs=%d D=%d H=%d L=%d A=%d (A + 1 <= %d)", d->B, d->D, d->H, d->L, d->A, HP);
  return mingru_rollout_step(*d, params, obs, state, out, (hipStream_t)stream);
}
