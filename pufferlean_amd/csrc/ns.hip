// Fused Newton-Schulz orthogonalisation of a batch of fp32 matrices on bf16 MFMA.
//
// One launch runs the whole quintic for every matrix of the batch: the Frobenius normalisation and
// all steps, with the iterate and its products resident in library scratch between phases (a few
// MB per matrix, so they stay in the L2 / Infinity Cache). Each matrix is taken in wide form
// (m = min(rows, cols) rows, w = max columns; tall inputs are transposed on the way in and out),
// zero-padded to multiples of 64, and each step
//   X' = aX + (bA + cA^2)X,   A = XX^T
// is evaluated in the shifted form, with E = A - I (so A^2 = I + 2E + E^2):
//   X' = (a+b+c)X + B'X,     B' = (b+2c)E + cE^2.
// It is the same polynomial, but the bf16 MFMA operands E and B' shrink as the singular values
// approach 1, so their rounding no longer cancels against the a*X term: at the same operand
// precision the shifted form roughly halves the error against an f64 iterate.
//
// Phases (each a list of 64x64 output tiles):
//   P0  raw input -> fp32, bf16 and transposed hi/lo bf16 wide copies; per-tile sums of squares
//   P1  E = s^2 XX^T - I       lower-triangle tiles (E is symmetric). Writes E in fp32 for the
//                              tile and its hi/lo bf16 halves (E = Eh + El) for the tile and its
//                              mirror, so later phases read whole rows
//   P2  B' = (b+2c)E + cE^2    lower-triangle tiles; E^2 = Eh Eh^T + Eh El^T + El Eh^T (three
//                              products of each k chunk's four panels). Writes the
//                              hi/lo bf16 halves of B' (tile and mirror)
//   P3  X' = s((a+b+c)X + B'X) all tiles; B'X = Bh Xh + Bh Xl + Bl Xh with X = Xh + Xl its hi/lo
//                              bf16 halves (three products likewise). Writes fp32, bf16 and
//                              transposed hi/lo bf16 copies of X', or the caller's matrix after
//                              the last step
// The lo half of X matters on real gradients: B' is O(1) while small singular values are still
// growing, and 5 steps amplify an error along a small singular direction up to a^5 ~ 480-fold, so
// B' times the bf16 rounding of X alone left 1.4-2.5e-2 on the MinGRU step's 1536x512 and 16x512
// momenta (an emulation of this arithmetic reproduces the measured errors); with it, <= 3e-3.
// s = 1/(||X||_F + eps) at step 0 (the copies hold the raw input), 1 afterwards. Zero padding is
// exact: padded rows/columns of X stay zero, and E's padded diagonal (-1) only meets zeros of X.
//
// Memory: every step has its own output buffers, so within a launch each address is written once,
// and only read after its writer has signalled. Those writes are device-coherent (write-through)
// stores, so a reader on another XCD finds them in memory, and no cache can hold a stale copy of a
// line that is read: nothing needs writing back or invalidating between phases, and operand reads
// keep the L2.
//
// Scheduling: every tile of every phase of every matrix is one work item with a ticket number in
// its matrix's queue, ordered by (step, phase, matrix, tile). An item waits only for the items of
// its matrix in earlier phases, all of them smaller tickets of the same queue. A queue's blocks take
// its tickets from an atomic counter in increasing order, so every item waited on has been taken by
// a block that is already running (or runs an earlier item of its own), and the launch completes for any
// grid size. Waits are bounded all the same. The launch's last block to leave resets the counters.
//
// Queues (ns_plan.hpp): on a device of 8 XCDs of 32 CUs (MI355X), one queue per XCD, served by the blocks that
// run on it (the XCC_ID hardware register), when every phase of every matrix fits one XCD (at most 32 tiles).
// Each matrix is pinned to one queue: its items, iterates and products stay on that XCD and the data moves
// through its L2 (plain stores, L2 hits; every line a block reads was written earlier in the launch by a
// block of the same XCD). Larger matrices and other devices take one device-wide queue, with
// device-coherent (write-through) stores. Control words are device-scope in both (atomics, and relaxed
// device-scope loads for polling; many blocks poll one word, and polling with atomics serialises them behind
// the signal they wait for). Measured (5 steps), pinned against device-wide: 200x129 119 us against
// 143, 256x256 125 / 155, 320x320 142 / 183, but 512x512 300 / 219 and 1536x512 592 / 287, hence the rule. The
// launch's last block checks that every queue with work had blocks on its XCD, else it raises a sticky
// flag that ph_ns_status reports.

#include "common.hpp"
#include "kernels.hpp"

#include <atomic>
#include <utility>

// The placements' instantiations give bit-identical matrices: every fused multiply-add is written out.
#pragma clang fp contract(off)

namespace ph {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));  // 8 bf16 (native vector: stays in VGPRs)

constexpr int kT = 64;          // output tile edge and k chunk
constexpr int kPitch = kT + 8;  // LDS row pitch in bf16 elements (144 B: conflict-free MFMA reads)
constexpr int kGroups = 2;      // k-groups per block: each takes every other k chunk of a tile
constexpr int kThreads = 256 * kGroups;  // a k-group is 4 wavefronts, one per 32x32 quadrant
constexpr int kSets1 = 4;       // k chunks in flight per k-group (register prefetch depth): one product
constexpr int kSets3 = 3;       // ... three products (four operand panels per chunk)
constexpr unsigned kSpinLimit = 1u << 20;  // bounded wait (about a second); never reached in a valid run

struct NsMat {
  float* x;           // caller's matrix, rows x cols, normalised and orthogonalised in place
  unsigned char* ws;  // this matrix's scratch (ns_layout)
  int rows, cols;
};

// Control words, each polled or updated on its own 128-byte line (32 words): the launch's blocks
// finished; the wait limit hit in this launch (kCtlFlag; +1: ever hit, +2: a queue with work had no
// blocks on its XCD, both never cleared by the kernel); the XCDs that had blocks in this launch (bit
// mask); per queue its next ticket; per matrix its items done.
constexpr int kCtlStride = 32;
constexpr int kCtlOut = 0;
constexpr int kCtlFlag = kCtlStride;
constexpr int kCtlSeen = 2 * kCtlStride;
constexpr int kCtlTicket = 3 * kCtlStride;                    // + kCtlStride * q
constexpr int kCtlDone = kCtlTicket + kCtlStride * kNsQueues;  // + kCtlStride * matrix
constexpr int kCtlWords = kCtlDone + kCtlStride * kNsMaxMats;

struct NsLaunch {
  NsMat mat[kNsMaxMats];
  NsItems i0, it, i3;
  float coef[3 * kNsMaxSteps];
  unsigned* ctl;  // control words (kCtl*)
  int nmat, nsteps, nq;
  float eps;
  unsigned spin;   // wait bound (polls)
  unsigned qmask;  // queues with work (bit q)
};

// Buffers of step s start at base + s * stride (x*: the step's input iterate, e*/b*: its E and B').
struct Geo {
  int m, w, mp, wp, tm, tw;
  bool tall;
  long n0, nt, n3;
  long mw, mm;  // per-step strides (elements) of the wide and the square buffers
  float *xf, *ef, *part;
  uint16_t *xb, *xt, *xtl, *eh, *el, *bh, *bl;
};

// Geometry and scratch layout of one matrix for nsteps steps; returns the scratch bytes it needs.
__host__ __device__ inline size_t ns_layout(int rows, int cols, int nsteps, unsigned char* base, Geo& g) {
  g.tall = rows > cols;
  g.m = g.tall ? cols : rows;
  g.w = g.tall ? rows : cols;
  g.tm = (g.m + kT - 1) / kT;
  g.tw = (g.w + kT - 1) / kT;
  g.mp = g.tm * kT;
  g.wp = g.tw * kT;
  g.n0 = (long)g.tm * g.tw;
  g.nt = (long)g.tm * (g.tm + 1) / 2;
  g.n3 = g.n0;
  g.mw = (long)g.mp * g.wp;  // multiples of 64 * 64 elements: every step's buffer stays aligned
  g.mm = (long)g.mp * g.mp;
  const size_t ns = (size_t)nsteps, mw = (size_t)g.mw, mm = (size_t)g.mm;
  size_t off = 0;
  auto take = [&](size_t bytes) {
    const size_t at = off;
    off += (bytes + 255) & ~(size_t)255;
    return (void*)((uintptr_t)base + at);
  };
  g.xf = (float*)take(4 * mw * ns);
  g.ef = (float*)take(4 * mm * ns);
  g.xb = (uint16_t*)take(2 * mw * ns);
  g.xt = (uint16_t*)take(2 * mw * ns);
  g.xtl = (uint16_t*)take(2 * mw * ns);
  g.eh = (uint16_t*)take(2 * mm * ns);
  g.el = (uint16_t*)take(2 * mm * ns);
  g.bh = (uint16_t*)take(2 * mm * ns);
  g.bl = (uint16_t*)take(2 * mm * ns);
  g.part = (float*)take(4 * (size_t)g.n0);
  return off;
}

__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Stores of every value another block reads in this launch. LOCAL (the reader runs on the same XCD):
// plain stores, which the write-through L1 passes to the XCD's L2. Otherwise device-coherent stores
// (relaxed agent-scope atomic stores: write-through to memory, sc1).
template <bool LOCAL, typename T>
__device__ __forceinline__ void st_dev(T* p, T v) {
  if constexpr (LOCAL) *p = v;
  else __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Control-word atomics and polls, device scope (see the scheduling notes).
__device__ __forceinline__ unsigned ctl_add(unsigned* p, unsigned v) {
  return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned ctl_load(unsigned* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void ctl_store(unsigned* p, unsigned v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Thread 0 waits until `need` items of the matrix are done (relaxed polls: the data they guard is
// read for the first time after the wait, from the L2 it was written to, or from memory). The wait
// is bounded: past the limit it raises the launch's flag, and once the flag is up no further wait
// blocks, so the launch always drains quickly (with wrong results) instead of hanging.
__device__ void wait_done(unsigned* cnt, unsigned need, unsigned* flag, unsigned limit) {
  if (threadIdx.x == 0) {
    unsigned spins = 0;
    while (ctl_load(cnt) < need && ctl_load(flag) == 0u) {
      __builtin_amdgcn_s_sleep(2);
      if (++spins > limit) {
        ctl_store(flag, 1u);
        ctl_store(flag + 1, 1u);  // sticky record
        break;
      }
    }
  }
  __syncthreads();
}

// Every thread's stores have completed, then the item counts as done. A completed store has reached
// the XCD's L2 (LOCAL: where the readers look) or memory (device-coherent stores), so no L2
// write-back (an agent-scope release fence) is needed, and none is paid for (it measured 5-15 us
// per item). The asm's memory clobber keeps the compiler from moving stores past the wait.
__device__ void signal_done(unsigned* cnt) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) ctl_add(cnt, 1u);
}

// s = 1/(sqrt(sum of the P0 partials) + eps), summed in the same fixed order by every wavefront.
__device__ float norm_scale(const float* part, long n0, float eps) {
  const int lane = threadIdx.x & 63;
  float v = 0.f;
  for (long i = lane; i < n0; i += 64) v += part[i];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return 1.f / (sqrtf(v) + eps);
}

// Lower-triangle tile index -> (ti, tj), ti >= tj, row-major over the triangle.
__device__ inline void tri_coords(long r, int& ti, int& tj) {
  int i = (int)((sqrtf(8.f * (float)r + 1.f) - 1.f) * 0.5f);
  while ((long)i * (i + 1) / 2 > r) i--;
  while ((long)(i + 1) * (i + 2) / 2 <= r) i++;
  ti = i;
  tj = (int)(r - (long)i * (i + 1) / 2);
}

// acc0 + acc1 = this k-group's share of A[64 rows][K] . B[64 rows][K]^T for this wavefront's 32x32 quadrant
// (wr, wc): k-group g takes the 64-wide k chunks g, g + kGroups, ... X3: the operands are hi/lo pairs
// (the lo half da / db elements behind the hi half) and the sum is Ah Bh + Ah Bl + Al Bh, each chunk's four
// panels read once for its three products (a k loop per product reads six: with one CU taking in
// 50-65 GB/s, the panels are what a three-product item costs). a / b point at the tile's first row; rows are ld apart;
// K is a multiple of 64. Chunks are loaded NS - 1 steps ahead into registers, staged through the group's
// double-buffered LDS, and read as one 16-byte fragment per lane per MFMA. Both groups run the same number
// of steps (block barriers stay matched); a step whose chunk is past the end only skips its MFMAs.
struct TileOps {
  const uint16_t *a, *b;
  long da, db;
  long ld;
  int K;
};
constexpr int kPanel = kT * kPitch;  // LDS elements of one staged 64x64 panel

template <bool X3, int NS, int... I>
__device__ __forceinline__ void mma_tile(const TileOps& op, uint16_t* lds, floatx16& acc0, floatx16& acc1,
                                         std::integer_sequence<int, I...>) {
  constexpr int NP = X3 ? 4 : 2;  // panels per chunk: Ah, Bh (, Al, Bl)
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int grp = wave >> 2, gw = wave & 3;
  const int wr = gw >> 1, wc = gw & 1;
  const int lr = lane & 31, lk = (lane >> 5) * 16;
  const int nc = op.K / kT;
  const int nsteps = (nc + kGroups - 1) / kGroups;
  uint16_t* const gl = lds + grp * 2 * NP * kPanel;  // this group's two buffers
  // this thread's two 16-byte pieces of each 64x64 panel
  const int gt = tid & 255, prow = gt >> 3, pk = (gt & 7) * 8;
  const long off = (long)prow * op.ld + pk, off32 = 32 * op.ld;
  const uint16_t* const src[4] = {op.a + off, op.b + off, op.a + op.da + off, op.b + op.db + off};
  u32x4 rg[NS][NP][2];
  auto gload = [&](u32x4 (&x)[NP][2], int i) __attribute__((always_inline)) {
    int c = i * kGroups + grp;
    c = c < nc ? c : nc - 1;  // past the end: reload the last chunk (never computed on)
#pragma unroll
    for (int p = 0; p < NP; p++)
#pragma unroll
      for (int h = 0; h < 2; h++) x[p][h] = *reinterpret_cast<const u32x4*>(src[p] + c * kT + h * off32);
  };
  auto sstore = [&](const u32x4 (&x)[NP][2], int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < NP; p++)
#pragma unroll
      for (int h = 0; h < 2; h++)
        *reinterpret_cast<u32x4*>(gl + (buf * NP + p) * kPanel + (prow + 32 * h) * kPitch + pk) = x[p][h];
  };
  auto mfma = [&](floatx16& c, const u32x4& a, const u32x4& b) __attribute__((always_inline)) {
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  };
  const int fa = (wr * 32 + lr) * kPitch + lk, fb = kPanel + (wc * 32 + lr) * kPitch + lk;
  auto compute = [&](int buf) __attribute__((always_inline)) {
    const uint16_t* base = gl + buf * NP * kPanel;
    auto rd = [&](int o) __attribute__((always_inline)) { return *reinterpret_cast<const u32x4*>(base + o); };
#pragma unroll
    for (int kb = 0; kb < kT; kb += 32) {
#pragma unroll
      for (int h = 0; h < 16; h += 8) {
        const u32x4 a = rd(fa + kb + h), b = rd(fb + kb + h);
        floatx16& c0 = h ? acc1 : acc0;
        mfma(c0, a, b);
        if constexpr (X3) {
          floatx16& c1 = h ? acc0 : acc1;
          const u32x4 al = rd(2 * kPanel + fa + kb + h), bl = rd(2 * kPanel + fb + kb + h);
          mfma(c1, a, bl);
          mfma(c0, al, b);
        }
      }
    }
  };
  for (int r = 0; r < 16; r++) acc0[r] = acc1[r] = 0.f;
  // prologue: chunks 0..NS-1 in flight, chunk 0 in LDS buffer 0
  (gload(rg[I], I), ...);
  sstore(rg[0], 0);
  lds_barrier();
  // step i (set S = i % NS): refill set S with step i + NS's chunk, compute step i's chunk, stage
  // step i + 1's
  auto step = [&](int i, auto Sc) __attribute__((always_inline)) {
    constexpr int S = decltype(Sc)::value, S1 = (S + 1) % NS;
    if (i >= nsteps) return;
    gload(rg[S], i + NS);
    __builtin_amdgcn_sched_barrier(0);
    if (i * kGroups + grp < nc) compute(i & 1);
    __builtin_amdgcn_sched_barrier(0);
    sstore(rg[S1], (i + 1) & 1);
    lds_barrier();
  };
  for (int i = 0; i < nsteps; i += NS) (step(i + I, std::integral_constant<int, I>{}), ...);
}

// Accumulator element e of this lane sits at tile row wr*32 + 8*(e/4) + 4*(lane/32) + e%4 and
// tile column wc*32 + lane%32.
__device__ __forceinline__ int acc_row(int e) {
  const int lane = threadIdx.x & 63, wr = ((threadIdx.x >> 6) & 3) >> 1;
  return wr * 32 + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
}
__device__ __forceinline__ int acc_col() {
  const int lane = threadIdx.x & 63, wc = ((threadIdx.x >> 6) & 3) & 1;
  return wc * 32 + (lane & 31);
}

// hi/lo bf16 halves of v (v = hi + lo to about 16 bits)
__device__ __forceinline__ void split_bf16(float v, uint16_t& h, uint16_t& l) {
  h = bf16_rne(v);
  l = bf16_rne(v - bf16_to_f32(h));
}

// Store the 4 consecutive-row values q*4..q*4+3 of this lane as 4 consecutive bf16 of the mirrored
// row (tile column -> row).
template <bool LOCAL>
__device__ __forceinline__ void store_mirror4(uint16_t* dst, const uint16_t (&v)[4]) {
  st_dev<LOCAL>(reinterpret_cast<uint64_t*>(dst), (uint64_t)v[0] | ((uint64_t)v[1] << 16) |
                                                      ((uint64_t)v[2] << 32) | ((uint64_t)v[3] << 48));
}

// P0: one 64x64 tile of the wide input into the fp32 / bf16 / transposed bf16 copies, plus the
// tile's sum of squares (fixed order).
template <bool LOCAL>
__device__ void p0_convert(const NsMat& mt, const Geo& g, long r, float* stage) {
  const int ti = (int)(r / g.tw), tj = (int)(r % g.tw);
  const int tid = threadIdx.x;
  // stage[a * 65 + b] = X_wide(ti*64 + a, tj*64 + b); loads run along the source's rows
  for (int it = 0; it < kT * kT / kThreads; it++) {
    const int id = it * kThreads + tid, a = id >> 6, b = id & 63;
    if (!g.tall) {
      const int wi = ti * kT + a, wj = tj * kT + b;
      stage[a * 65 + b] = (wi < g.m && wj < g.w) ? mt.x[(long)wi * mt.cols + wj] : 0.f;
    } else {
      const int wj = tj * kT + a, wi = ti * kT + b;  // source row wj, column wi
      stage[b * 65 + a] = (wi < g.m && wj < g.w) ? mt.x[(long)wj * mt.cols + wi] : 0.f;
    }
  }
  __syncthreads();
  float ss = 0.f;
  for (int it = 0; it < kT * kT / kThreads; it++) {
    const int id = it * kThreads + tid, a = id >> 6, b = id & 63;
    const float v = stage[a * 65 + b];
    ss = fmaf(v, v, ss);
    const long o = (long)(ti * kT + a) * g.wp + tj * kT + b;
    st_dev<LOCAL>(&g.xf[o], v);
    st_dev<LOCAL>(&g.xb[o], bf16_rne(v));
    uint16_t th, tl;
    split_bf16(stage[b * 65 + a], th, tl);
    const long ot = (long)(tj * kT + a) * g.mp + ti * kT + b;
    st_dev<LOCAL>(&g.xt[ot], th);
    st_dev<LOCAL>(&g.xtl[ot], tl);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o);
  __syncthreads();
  if ((tid & 63) == 0) stage[tid >> 6] = ss;
  __syncthreads();
  if (tid == 0) {
    float t = 0.f;
    for (int w = 0; w < kThreads / 64; w++) t += stage[w];
    st_dev<LOCAL>(&g.part[r], t);
  }
}

// P3's epilogue of NE accumulator elements of this lane: element e (value v[e] = (B'X)(row, col), old iterate
// pre[e]) at row rb + 8 (e / 4) + e % 4, column col of the wide matrix.
template <bool LOCAL, int NE>
__device__ __forceinline__ void p3_store(const NsMat& mt, const Geo& g, long xs, int rb, int col, const float (&v)[NE],
                                         const float (&pre)[NE], float abc, float sc, bool last) {
  float* xfn = g.xf + xs + g.mw;  // next step's input (not touched after the last step)
  uint16_t* xbn = g.xb + xs + g.mw;
  uint16_t* xtn = g.xt + xs + g.mw;
  uint16_t* xtln = g.xtl + xs + g.mw;
#pragma unroll
  for (int q = 0; q < NE / 4; q++) {
    uint16_t x4[4], l4[4];
#pragma unroll
    for (int e4 = 0; e4 < 4; e4++) {
      const int row = rb + 8 * q + e4;
      const long o = (long)row * g.wp + col;
      const float x = sc * fmaf(abc, pre[4 * q + e4], v[4 * q + e4]);
      if (last) {
        if (row < g.m && col < g.w) {
          if (g.tall) mt.x[(long)col * mt.cols + row] = x;
          else mt.x[(long)row * mt.cols + col] = x;
        }
      } else {
        st_dev<LOCAL>(&xfn[o], x);
        split_bf16(x, x4[e4], l4[e4]);
        st_dev<LOCAL>(&xbn[o], x4[e4]);
      }
    }
    if (!last) {
      const long om = (long)col * g.mp + rb + 8 * q;
      store_mirror4<LOCAL>(xtn + om, x4);
      store_mirror4<LOCAL>(xtln + om, l4);
    }
  }
}

// LOCAL: every matrix's items run on one XCD (plain stores), a block serving the queue of the XCD it runs on;
// otherwise one device-wide queue and device-coherent stores.
template <bool LOCAL>
__global__ void __launch_bounds__(kThreads) k_ns_fused(const NsLaunch L) {
  // the two k-groups' double-buffered panels; the epilogue's fold and P0's staging reuse them
  __shared__ __align__(16) uint16_t lds[kGroups * 2 * 4 * kPanel];
  __shared__ unsigned s_ticket;
  static_assert(sizeof(lds) + 16 <= 160 * 1024, "LDS budget (one block per CU)");
  unsigned* ctl = L.ctl;
  const int tid = threadIdx.x;
  int qi = 0;
  if (L.nq > 1) {
    unsigned xcc;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcc));
    qi = (int)(xcc & 0xfu);
  }
  if (tid == 0 && qi < kNsQueues)
    __hip_atomic_fetch_or(&ctl[kCtlSeen], 1u << qi, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (qi >= L.nq) qi = -1;  // not a queue's XCD: no work (the last block checks coverage)
  const int qc = qi < 0 ? 0 : qi;
  const int lo0 = L.i0.qlo[qc], lot = L.it.qlo[qc], lo3 = L.i3.qlo[qc];
  const int n0q = L.i0.qlo[qc + 1] - lo0, ntq = L.it.qlo[qc + 1] - lot, n3q = L.i3.qlo[qc + 1] - lo3;
  const int total = qi < 0 ? 0 : n0q + L.nsteps * (2 * ntq + n3q);
  unsigned* const tick = &ctl[kCtlTicket + kCtlStride * qc];
  if (tid == 0) s_ticket = total > 0 ? ctl_add(tick, 1u) : 0u;
  __syncthreads();
  int t = (int)s_ticket;
  // tickets only grow: the phase of the current one is found by walking forward. Phase (p, s) holds the
  // queue's tickets [pbeg, pbeg + pcnt).
  int p = 0, s = 0, pbeg = 0, pcnt = n0q;
  for (; t < total; t = (int)s_ticket) {
    while (t >= pbeg + pcnt) {
      pbeg += pcnt;
      if (p == 3) { p = 1; s++; }
      else p++;
      pcnt = p == 3 ? n3q : ntq;
    }
    const NsItems& im = p == 0 ? L.i0 : (p == 3 ? L.i3 : L.it);
    int r = t - pbeg + (p == 0 ? lo0 : (p == 3 ? lo3 : lot));
    int gi = 0;
    while (gi < L.nmat - 1 && r >= im.cum[gi + 1]) gi++;
    r -= im.cum[gi];
    const NsMat mt = L.mat[gi];  // a copy: a reference would move the kernel argument to scratch
    Geo g;
    ns_layout(mt.rows, mt.cols, L.nsteps, mt.ws, g);
    unsigned* const done = &ctl[kCtlDone + kCtlStride * gi];
    // The next ticket is taken while this item runs (its round trip overlaps the stores' drain). Still
    // in order: an item's ticket is held by a block that runs it or an earlier one, and items wait only
    // for earlier phases, so the earliest unfinished item is always running or next on its block.
    unsigned next = 0u;
    if (p == 0) {
      if (tid == 0) next = ctl_add(tick, 1u);
      p0_convert<LOCAL>(mt, g, r, reinterpret_cast<float*>(lds));
      if (tid == 0) s_ticket = next;
      signal_done(done);
      continue;
    }
    const long need = g.n0 + (long)s * (2 * g.nt + g.n3) + (p - 1) * g.nt;
    wait_done(done, (unsigned)need, &ctl[kCtlFlag], L.spin);
    const float a = L.coef[3 * s], b = L.coef[3 * s + 1], c = L.coef[3 * s + 2];
    const float sc = s == 0 ? norm_scale(g.part, g.n0, L.eps) : 1.f;
    const long xs = (long)s * g.mw, es = (long)s * g.mm;  // this step's buffers
    int ti, tj;
    TileOps op;
    if (p == 3) {
      // column by column: blocks that run side by side share rows of X^T and, as m <= w, read at most all of B'
      tj = r / g.tm;
      ti = r - tj * g.tm;
      op.ld = g.mp;
      op.K = g.mp;
      // A: B' = (Bh, Bl) rows ti; B: X^T = (Xh^T, Xl^T) rows tj
      op.a = g.bh + es + (long)ti * kT * g.mp;
      op.da = g.bl - g.bh;
      op.b = g.xt + xs + (long)tj * kT * g.mp;
      op.db = g.xtl - g.xt;
    } else {
      tri_coords(r, ti, tj);
      if (p == 1) {
        op.ld = g.wp;
        op.K = g.wp;
        op.a = g.xb + xs + (long)ti * kT * g.wp;
        op.b = g.xb + xs + (long)tj * kT * g.wp;
        op.da = op.db = 0;
      } else {
        op.ld = g.mp;
        op.K = g.mp;
        // A: E = (Eh, El) rows ti; B: E rows tj
        op.a = g.eh + es + (long)ti * kT * g.mp;
        op.b = g.eh + es + (long)tj * kT * g.mp;
        op.da = op.db = g.el - g.eh;
      }
    }
    // Both k-groups run the epilogue, each on half of the quadrant's rows (accumulator elements
    // e0 .. e0 + 7). Its fp32 operand (E for P2, X for P3) is loaded before the k loop, so that its memory
    // latency overlaps the products.
    const int e0 = 8 * (tid >> 8);
    float pre[8];
    if (p >= 2) {
      const float* src = p == 2 ? g.ef + es : g.xf + xs;
      const long ld = p == 2 ? g.mp : g.wp;
      const int c0 = tj * kT + acc_col(), r0 = ti * kT;
#pragma unroll
      for (int e = 0; e < 8; e++) pre[e] = src[(long)(r0 + acc_row(e0 + e)) * ld + c0];
    }
    floatx16 acc0, acc1;
    if (p == 1) mma_tile<false, kSets1>(op, lds, acc0, acc1, std::make_integer_sequence<int, kSets1>{});
    else mma_tile<true, kSets3>(op, lds, acc0, acc1, std::make_integer_sequence<int, kSets3>{});
    if (tid == 0) next = ctl_add(tick, 1u);
    // fold the two k-groups' partial tiles: each hands the other's half over through LDS
    float* red = reinterpret_cast<float*>(lds);
    float v8[8];
    {
      float mine[16];
#pragma unroll
      for (int e = 0; e < 16; e++) mine[e] = acc0[e] + acc1[e];
      const bool hi = tid >= 256;
#pragma unroll
      for (int e = 0; e < 8; e++) red[e * kThreads + tid] = hi ? mine[e] : mine[8 + e];
      __syncthreads();
#pragma unroll
      for (int e = 0; e < 8; e++) v8[e] = (hi ? mine[8 + e] : mine[e]) + red[e * kThreads + (tid ^ 256)];
    }
    const int col = tj * kT + acc_col();
    const int row0 = ti * kT;
    if (p != 3) {
      uint16_t* hi = (p == 1 ? g.eh : g.bh) + es;
      uint16_t* lo = (p == 1 ? g.el : g.bl) + es;
      float* ef = g.ef + es;
      const float cE = b + 2.f * c;
#pragma unroll
      for (int q = 0; q < 2; q++) {
        uint16_t h4[4], l4[4];
#pragma unroll
        for (int e4 = 0; e4 < 4; e4++) {
          const int e = 4 * q + e4;
          const int row = row0 + acc_row(e0 + e);
          const long o = (long)row * g.mp + col;
          const float v = v8[e];
          float val;
          if (p == 1) {
            val = fmaf(sc * sc, v, row == col ? -1.f : 0.f);
            st_dev<LOCAL>(&ef[o], val);
          } else {
            val = fmaf(cE, pre[e], c * v);
          }
          split_bf16(val, h4[e4], l4[e4]);
          st_dev<LOCAL>(&hi[o], h4[e4]);
          st_dev<LOCAL>(&lo[o], l4[e4]);
        }
        if (ti != tj) {
          const long om = (long)col * g.mp + row0 + acc_row(e0 + 4 * q);
          store_mirror4<LOCAL>(hi + om, h4);
          store_mirror4<LOCAL>(lo + om, l4);
        }
      }
    } else {
      p3_store<LOCAL, 8>(mt, g, xs, row0 + acc_row(e0), col, v8, pre, a + b + c, sc, s == L.nsteps - 1);
    }
    if (tid == 0) s_ticket = next;
    signal_done(done);
  }
  // Leave. The launch's last block out (every other block has taken its final ticket and finished
  // its items) checks that every queue with work had blocks on its XCD and resets the counters.
  if (tid == 0) {
    const unsigned out = __hip_atomic_fetch_add(&ctl[kCtlOut], 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
    if (out == gridDim.x - 1) {
      if ((L.qmask & ~ctl_load(&ctl[kCtlSeen])) != 0u) ctl_store(&ctl[kCtlFlag + 2], 1u);
      ctl_store(&ctl[kCtlSeen], 0u);
      ctl_store(&ctl[kCtlFlag], 0u);
      for (int q = 0; q < L.nq; q++) ctl_store(&ctl[kCtlTicket + kCtlStride * q], 0u);
      for (int i = 0; i < L.nmat; i++) ctl_store(&ctl[kCtlDone + kCtlStride * i], 0u);
      __hip_atomic_store(&ctl[kCtlOut], 0u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

// ---- small matrices: the whole iteration in one workgroup's LDS ------------------------------------------
// A matrix whose X^T and E (hi and lo bf16 halves) fit the 160 KB of one CU runs every phase of every step
// in one block: the phases are separated by workgroup barriers instead of write-through stores, a signal and
// a poll through memory, which cost k_ns_fused 6-7 us a phase on such a matrix whatever its size. Bound by the
// LDS reads of the three-product phases (4 KB per 32x32x16 step) and the barriers. X and E stay in fp32 in the
// accumulator registers of the wavefront that owns the tile. The CartPole policy's three matrices (128x128,
// 128x4, 3x128), five steps: 105 -> 62 us, one block each.
// Every element sees k_ns_fused's operands and order: k chunks of 64 in two groups by parity, the groups'
// sums of two accumulators each, the lower 64x64 blocks of E^2 mirrored, the norm from 64x64 tile sums. So
// the matrices are bit-identical to its, and a small matrix gives the same result alone and in a batch with
// large ones.
constexpr int kSmallEl = (160 * 1024 - 512) / 2;  // LDS elements (bf16) for X^T and E
constexpr int kSmallTiles = 16;                   // 32x32 tiles of X: two per wavefront (four spill)
struct NsSmall {
  float* x[kNsMaxMats];
  int rows[kNsMaxMats], cols[kNsMaxMats];
  float coef[3 * kNsMaxSteps];
  int nsteps;
  float eps;
};
struct SmallGeo {
  int m, w, tm, tw;  // wide form, and its extents in 32x32 tiles
  int pm;            // LDS row pitch (elements): rows 4 (mod 8) 16-byte pieces apart
  bool tall;
};
__host__ __device__ inline SmallGeo small_geo(int rows, int cols) {
  SmallGeo g;
  g.tall = rows > cols;
  g.m = g.tall ? cols : rows;
  g.w = g.tall ? rows : cols;
  g.tm = (g.m + 31) / 32;
  g.tw = (g.w + 31) / 32;
  g.pm = g.tm * 32 + 8;
  return g;
}
inline bool small_fits(int rows, int cols) {
  const int mn = rows < cols ? rows : cols, mx = rows < cols ? cols : rows;
  if (mn > 128 || mx > 1024) return false;
  const SmallGeo g = small_geo(rows, cols);
  return g.tm * g.tw <= kSmallTiles && 2 * g.pm * 32 * (g.tw + g.tm) <= kSmallEl;
}

// 8 consecutive k (rows k0.. of a [k][pm] array) at column c0 + lane % 32, k0 the lane's own: two transposing
// reads of every other row (distinct banks at this pitch) interleaved back into k order.
typedef short ns_v4i16 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u32x4 small_tr(const uint16_t* a, int pm, int c0, int k0, int lane) {
  const int sl = lane & 15, c = c0 + ((lane >> 4) & 1) * 16 + 4 * (sl & 3);
  uint32_t w[2][2];
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const uint16_t* p = a + (k0 + 2 * (sl >> 2) + h) * pm + c;
    const ns_v4i16 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) ns_v4i16*)(__attribute__((address_space(3))) void*)p);
    w[h][0] = (uint32_t)(uint16_t)v[0] | ((uint32_t)(uint16_t)v[1] << 16);
    w[h][1] = (uint32_t)(uint16_t)v[2] | ((uint32_t)(uint16_t)v[3] << 16);
  }
  u32x4 r;
#pragma unroll
  for (int q = 0; q < 2; q++) {
    r[2 * q] = (w[0][q] & 0xffffu) | (w[1][q] << 16);
    r[2 * q + 1] = (w[0][q] >> 16) | (w[1][q] & 0xffff0000u);
  }
  return r;
}

template <int NU>  // tiles of X per wavefront
__global__ void __launch_bounds__(512) k_ns_small(const NsSmall L) {
  __shared__ __align__(16) uint16_t sm[kSmallEl];
  __shared__ float red[64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int rows = L.rows[blockIdx.x], cols = L.cols[blockIdx.x];
  float* const x = L.x[blockIdx.x];
  const SmallGeo g = small_geo(rows, cols);
  const int pm = g.pm, mp = g.tm * 32, wp = g.tw * 32;
  uint16_t* const xh = sm;            // X^T hi, lo: [wp][pm]
  uint16_t* const xl = xh + wp * pm;
  uint16_t* const eh = xl + wp * pm;  // E, then B', hi, lo: [mp][pm]
  uint16_t* const el = eh + mp * pm;
  int hrow = 4 * (lane >> 5), lcol = lane & 31;
  int lr = lane & 31, lk = (lane >> 5) * 16;
  // keeps the compiler from computing a phase's addresses ahead of it and holding them across the others
  // (some 500 registers of them)
  auto fresh = [&]() __attribute__((always_inline)) {
    asm volatile("" : "+v"(hrow), "+v"(lcol), "+v"(lr), "+v"(lk));
  };
  auto at = [&](int i, int j) { return g.tall ? (long)j * cols + i : (long)i * cols + j; };  // wide (i, j) in x
  auto trow = [&](int t0, int e) { return t0 * 32 + 8 * (e >> 2) + hrow + (e & 3); };

  // this wavefront's tiles of X (tile wave + 8 u, column by column) in accumulator layout
  float xr[NU][16];
#pragma unroll
  for (int u = 0; u < NU; u++) {
    const int t = wave + 8 * u, tj = t / g.tm, ti = t - tj * g.tm;
#pragma unroll
    for (int e = 0; e < 16; e++) {
      const int i = trow(ti, e), j = tj * 32 + lcol;
      xr[u][e] = tj < g.tw && i < g.m && j < g.w ? x[at(i, j)] : 0.f;
    }
    fresh();
  }
  // 1 / (norm + eps): sums of squares by 64x64 tiles, in P0's order
  float sc0;
  {
    const int tm64 = (g.m + 63) / 64, tw64 = (g.w + 63) / 64, n0 = tm64 * tw64;
    for (int r = 0; r < n0; r++) {
      const int ti = r / tw64, tj = r - ti * tw64;
      float v[8], ss = 0.f;
#pragma unroll
      for (int it = 0; it < 8; it++) {
        const int i = ti * 64 + it * 8 + wave, j = tj * 64 + lane;
        v[it] = i < g.m && j < g.w ? x[at(i, j)] : 0.f;
      }
#pragma unroll
      for (int it = 0; it < 8; it++) ss = fmaf(v[it], v[it], ss);
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o);
      if (lane == 0) red[wave] = ss;
      __syncthreads();
      if (tid == 0) {
        float t = 0.f;
        for (int w = 0; w < 8; w++) t += red[w];
        red[16 + r] = t;
      }
      __syncthreads();
    }
    float v = lane < n0 ? red[16 + lane] : 0.f;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    sc0 = 1.f / (sqrtf(v) + L.eps);
  }
  auto mfma = [&](floatx16& c, const u32x4& a, const u32x4& b) __attribute__((always_inline)) {
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  };
  auto ld = [&](const uint16_t* p) __attribute__((always_inline)) { return *reinterpret_cast<const u32x4*>(p); };
  // acc[chunk parity][h] over nk 32-wide k blocks: body(accumulators, k, h) for each half
  auto kloop = [&](floatx16 (&acc)[2][2], int nk, auto body) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[q >> 1][q & 1][r] = 0.f;
    for (int it = 0; it < nk; it += 4) {
#pragma unroll
      for (int q = 0; q < 4; q++) {
        if (it + q >= nk) break;
        const int k = (it + q) * 32 + lk;
        body(acc[q >> 1][0], acc[q >> 1][1], k);
        body(acc[q >> 1][1], acc[q >> 1][0], k + 8);
        __builtin_amdgcn_sched_barrier(0);  // bounds the fragments in flight (registers)
      }
    }
  };
  // Ah Bh + Ah Bl + Al Bh of rows ar of (ah, al) and rows br of (bh, bl)
  auto prod3 = [&](floatx16 (&acc)[2][2], const uint16_t* ah, const uint16_t* al, int ar, const uint16_t* bh,
                   const uint16_t* bl, int br, int nk) __attribute__((always_inline)) {
    const int oa = (ar + lr) * pm, ob = (br + lr) * pm;
    kloop(acc, nk, [&](floatx16& c0, floatx16& c1, int k) __attribute__((always_inline)) {
      const u32x4 a = ld(ah + oa + k), b = ld(bh + ob + k), a2 = ld(al + oa + k), b2 = ld(bl + ob + k);
      mfma(c0, a, b);
      mfma(c1, a, b2);
      mfma(c0, a2, b);
    });
  };
  // a tile's 16 values into the E / B' arrays at (row, col) and, below the 64x64 diagonal, mirrored
  auto put_sq = [&](int ti, int tj, const float (&v)[16]) __attribute__((always_inline)) {
    const int col = tj * 32 + lcol;
#pragma unroll
    for (int q = 0; q < 4; q++) {
      uint16_t h4[4], l4[4];
      const int r0 = trow(ti, 4 * q);
#pragma unroll
      for (int e = 0; e < 4; e++) {
        split_bf16(v[4 * q + e], h4[e], l4[e]);
        eh[(r0 + e) * pm + col] = h4[e];
        el[(r0 + e) * pm + col] = l4[e];
      }
      if ((ti >> 1) > (tj >> 1)) {
        store_mirror4<true>(eh + col * pm + r0, h4);
        store_mirror4<true>(el + col * pm + r0, l4);
      }
    }
  };
  auto put_x = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < NU; u++) {
      const int t = wave + 8 * u, tj = t / g.tm, ti = t - tj * g.tm;
      if (tj >= g.tw) break;
      fresh();
      const int col = tj * 32 + lcol;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        uint16_t h4[4], l4[4];
#pragma unroll
        for (int e = 0; e < 4; e++) split_bf16(xr[u][4 * q + e], h4[e], l4[e]);
        const int r0 = trow(ti, 4 * q);
        store_mirror4<true>(xh + col * pm + r0, h4);
        store_mirror4<true>(xl + col * pm + r0, l4);
      }
    }
  };

  fresh();
  put_x();
  __syncthreads();
  const int ne = g.tm * g.tm;  // tiles of E (at most 16: two per wavefront); above the 64x64 diagonal: mirrored
  for (int s = 0; s < L.nsteps; s++) {
    const float a = L.coef[3 * s], b = L.coef[3 * s + 1], c = L.coef[3 * s + 2];
    const float sc = s == 0 ? sc0 : 1.f, abc = a + b + c, cE = b + 2.f * c;
    float er[2][16];
    floatx16 acc[2][2];
    // P1 (the previous step's B' has been read: barrier before put_x)
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const int t = wave + 8 * u, ti = t / g.tm, tj = t - ti * g.tm;
      if (t >= ne || (ti >> 1) < (tj >> 1)) continue;
      fresh();
      kloop(acc, g.tw, [&](floatx16& c0, floatx16&, int k) __attribute__((always_inline)) {
        mfma(c0, small_tr(xh, pm, ti * 32, k, lane), small_tr(xh, pm, tj * 32, k, lane));
      });
#pragma unroll
      for (int e = 0; e < 16; e++) {
        const float v = (acc[0][0][e] + acc[0][1][e]) + (acc[1][0][e] + acc[1][1][e]);
        er[u][e] = fmaf(sc * sc, v, trow(ti, e) == tj * 32 + lcol ? -1.f : 0.f);
      }
      fresh();
      put_sq(ti, tj, er[u]);
    }
    __syncthreads();
    // P2
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const int t = wave + 8 * u, ti = t / g.tm, tj = t - ti * g.tm;
      if (t >= ne || (ti >> 1) < (tj >> 1)) continue;
      fresh();
      prod3(acc, eh, el, ti * 32, eh, el, tj * 32, g.tm);
#pragma unroll
      for (int e = 0; e < 16; e++) {
        const float v = (acc[0][0][e] + acc[0][1][e]) + (acc[1][0][e] + acc[1][1][e]);
        er[u][e] = fmaf(cE, er[u][e], c * v);
      }
    }
    __syncthreads();  // E has been read
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const int t = wave + 8 * u, ti = t / g.tm, tj = t - ti * g.tm;
      fresh();
      if (t < ne && (ti >> 1) >= (tj >> 1)) put_sq(ti, tj, er[u]);
    }
    __syncthreads();
    // P3
#pragma unroll
    for (int u = 0; u < NU; u++) {
      const int t = wave + 8 * u, tj = t / g.tm, ti = t - tj * g.tm;
      if (tj >= g.tw) break;
      fresh();
      prod3(acc, eh, el, ti * 32, xh, xl, tj * 32, g.tm);
#pragma unroll
      for (int e = 0; e < 16; e++) {
        const float v = (acc[0][0][e] + acc[0][1][e]) + (acc[1][0][e] + acc[1][1][e]);
        xr[u][e] = sc * fmaf(abc, xr[u][e], v);
      }
    }
    if (s + 1 < L.nsteps) {
      __syncthreads();  // X and B' have been read
      fresh();
      put_x();
      __syncthreads();
    }
  }
#pragma unroll
  for (int u = 0; u < NU; u++) {
    const int t = wave + 8 * u, tj = t / g.tm, ti = t - tj * g.tm;
    fresh();
#pragma unroll
    for (int e = 0; e < 16; e++) {
      const int i = trow(ti, e), j = tj * 32 + lcol;
      if (tj < g.tw && i < g.m && j < g.w) x[at(i, j)] = xr[u][e];
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// The batch in launches of up to kNsMaxMats blocks (every matrix fits).
int ns_small(float* const* X, const int* rows, const int* cols, int n, const float* coeffs, int nsteps, float eps,
             hipStream_t st) {
  NsSmall L{};
  for (int k = 0; k < 3 * nsteps; k++) L.coef[k] = coeffs[k];
  L.nsteps = nsteps;
  L.eps = eps;
  int i = 0;
  while (i < n) {
    int nm = 0, tiles = 0;
    for (; i < n && nm < kNsMaxMats; i++) {
      if ((long)rows[i] * cols[i] == 0) continue;
      L.x[nm] = X[i];
      L.rows[nm] = rows[i];
      L.cols[nm++] = cols[i];
      const SmallGeo g = small_geo(rows[i], cols[i]);
      if (g.tm * g.tw > tiles) tiles = g.tm * g.tw;
    }
    if (nm == 0) continue;
    if (tiles <= 8) k_ns_small<1><<<nm, 512, 0, st>>>(L);
    else k_ns_small<2><<<nm, 512, 0, st>>>(L);
    PH_LAUNCH_CHECK();
  }
  return PH_OK;
}

std::atomic<unsigned> g_spin{kSpinLimit};
// 0: by shape (one workgroup per matrix, one XCD per matrix, or one device-wide queue); 1: always one device-wide
// queue; 2: one XCD per matrix whenever the device has 8 XCDs of 32 CUs
std::atomic<int> g_queues{0};

__global__ void k_clear_word(unsigned* w) {
  if (threadIdx.x == 0) *w = 0u;
}

int cu_count() {
  static int n[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (n[dev] == 0) {
    int v = 0;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v <= 0) v = 256;
    n[dev] = v;
  }
  return n[dev];
}

}  // namespace

size_t ns_fused_ws_bytes(int rows, int cols, int nsteps) {
  Geo g;
  return ns_layout(rows, cols, nsteps, nullptr, g);
}

int ns_fused(float* const* X, const int* rows, const int* cols, int n, const float* coeffs, int nsteps,
             float eps, int ws_slot, int ctl_slot, hipStream_t st) {
  if (nsteps < 1 || nsteps > kNsMaxSteps) {
    set_error("newton_schulz (fused): steps must be in 1..%d", kNsMaxSteps);
    return PH_ERR_UNSUPPORTED;
  }
  const int mode = g_queues.load(std::memory_order_relaxed);
  // every matrix in one CU's LDS: no waits between workgroups at all (a forced placement runs the queues)
  bool small = mode == 0;
  for (int j = 0; j < n && small; j++) small = (long)rows[j] * cols[j] == 0 || small_fits(rows[j], cols[j]);
  if (small) return ns_small(X, rows, cols, n, coeffs, nsteps, eps, st);
  unsigned* ctl = (unsigned*)scratch(ctl_slot, kCtlWords * 4);
  if (!ctl) return PH_ERR_NOMEM;
  PH_TRY(ensure_zeroed_words(ctl, kCtlWords, st));
  // On a device of kNsQueues XCDs of kXcdCus CUs: matrices pinned to one XCD each when every phase of every
  // matrix fits it (one block per CU, so kXcdCus tiles at a time). Otherwise, and in mode 1, one device-wide
  // queue.
  const int cus = cu_count();
  bool local = mode != 1 && cus == kNsQueues * kXcdCus;
  if (local && mode == 0)
    for (int j = 0; j < n; j++) {
      Geo g;
      ns_layout(rows[j], cols[j], nsteps, nullptr, g);
      if (g.n3 > kXcdCus || g.nt > kXcdCus) local = false;
    }
  int i = 0;
  while (i < n) {
    // next group of at most kNsMaxMats non-empty matrices
    NsLaunch L{};
    size_t bytes = 0;
    NsMat mats[kNsMaxMats];
    NsLoad load[kNsMaxMats];
    int j = i;
    for (; j < n && L.nmat < kNsMaxMats; j++) {
      if ((long)rows[j] * cols[j] == 0) continue;
      const int k = L.nmat++;
      NsMat& m = mats[k];
      m.x = X[j];
      m.rows = rows[j];
      m.cols = cols[j];
      Geo g;
      const size_t b = ns_layout(rows[j], cols[j], nsteps, nullptr, g);
      m.ws = (unsigned char*)(uintptr_t)bytes;  // offset for now
      bytes += b;
      // tile-chunk products of a step: P1 over w, P2 three over m, P3 three over m
      const long cw = g.wp / kT, cm = g.mp / kT;
      load[k] = NsLoad{g.n0, g.nt, g.n3, g.n0 + (long)nsteps * (g.nt * cw + 3 * g.nt * cm + 3 * g.n3 * cm)};
    }
    i = j;
    if (L.nmat == 0) continue;
    unsigned char* ws = (unsigned char*)scratch(ws_slot, bytes);
    if (!ws) return PH_ERR_NOMEM;
    NsPlan plan;
    if (!ns_place(load, L.nmat, nsteps, local, plan)) {
      set_error("newton_schulz (fused): batch too large");
      return PH_ERR_UNSUPPORTED;
    }
    for (int k = 0; k < L.nmat; k++) {
      L.mat[k] = mats[plan.order[k]];
      L.mat[k].ws = ws + (uintptr_t)L.mat[k].ws;
    }
    L.i0 = plan.i0;
    L.it = plan.it;
    L.i3 = plan.i3;
    L.nq = plan.nq;
    const long total = (long)L.i0.cum[L.nmat] + (long)nsteps * (2L * L.it.cum[L.nmat] + L.i3.cum[L.nmat]);
    for (int k = 0; k < 3 * nsteps; k++) L.coef[k] = coeffs[k];
    L.ctl = ctl;
    L.nsteps = nsteps;
    L.eps = eps;
    L.spin = g_spin.load(std::memory_order_relaxed);
    // one block per CU: measured faster than two (half as many blocks polling, and a CU's load
    // bandwidth goes to one tile at a time). Per-XCD queues take every CU (a queue with no items releases
    // its blocks at once).
    const long cap = cus;
    const unsigned grid = local ? (unsigned)cap : (unsigned)(total < cap ? total : cap);
    L.qmask = 0u;
    for (int q = 0; q < L.nq; q++)
      if (L.i0.qlo[q + 1] > L.i0.qlo[q] || L.it.qlo[q + 1] > L.it.qlo[q] || L.i3.qlo[q + 1] > L.i3.qlo[q])
        L.qmask |= 1u << q;
    if (local) k_ns_fused<true><<<grid, kThreads, 0, st>>>(L);
    else k_ns_fused<false><<<grid, kThreads, 0, st>>>(L);
    PH_LAUNCH_CHECK();
  }
  return PH_OK;
}

}  // namespace ph

using namespace ph;

extern "C" int ph_ns_status(void* stream) {
  const hipStream_t st = as_stream(stream);
  PH_CHECK_HIP(hipStreamSynchronize(st));
  unsigned* ctl = (unsigned*)scratch_peek(kSlotNsCtl);
  if (!ctl) return PH_OK;  // no fused launch has run on this device
  unsigned rec[2] = {0u, 0u};
  PH_CHECK_HIP(hipMemcpy(rec, ctl + kCtlFlag + 1, sizeof(rec), hipMemcpyDeviceToHost));
  if (rec[0] == 0u && rec[1] == 0u) return PH_OK;
  if (rec[0]) k_clear_word<<<1, 64, 0, st>>>(ctl + kCtlFlag + 1);
  if (rec[1]) k_clear_word<<<1, 64, 0, st>>>(ctl + kCtlFlag + 2);
  PH_LAUNCH_CHECK();
  PH_CHECK_HIP(hipStreamSynchronize(st));
  if (rec[1])
    set_error("newton_schulz (fused): a workgroup ran on another XCD than its work queue's (the device does "
              "not dispatch workgroups to XCDs round-robin); the matrices written by the launches since the "
              "last status check are invalid; ph_ns_set_queues(1) selects the device-wide queue");
  else
    set_error("newton_schulz (fused): a bounded wait for another workgroup's tiles gave up; the matrices "
              "written by the launches since the last status check are invalid");
  return PH_ERR_HIP;
}

extern "C" int ph_ns_set_spin_limit(unsigned polls) {
  g_spin.store(polls ? polls : kSpinLimit, std::memory_order_relaxed);
  return PH_OK;
}

extern "C" int ph_ns_set_queues(int mode) {
  if (mode < 0 || mode > 2) {
    set_error("ph_ns_set_queues: mode must be 0 (by shape), 1 (device-wide) or 2 (per XCD)");
    return PH_ERR_ARG;
  }
  g_queues.store(mode, std::memory_order_relaxed);
  return PH_OK;
}
