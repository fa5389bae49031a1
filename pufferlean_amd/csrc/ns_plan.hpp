// Placement of a fused Newton-Schulz launch's work items on its queues (host code, no device types).
//
// The items of one phase kind (P0; P1 and P2; P3) are numbered through the launch's matrices in list order, and
// a queue owns a contiguous range of each kind. Every matrix belongs to one queue, so an item waits only for
// items of earlier phases of its own queue: smaller tickets, each taken by a block that runs it or an earlier
// one. The launch therefore completes for any set of blocks that reaches every queue with work, in whatever
// order and number they start. Dealing one matrix's items over several queues would break that: blocks
// of one XCD would wait for blocks of another, which a kernel on another stream or process can hold back.
#pragma once
#include <utility>

namespace ph {

constexpr int kNsMaxMats = 16;  // matrices per launch
constexpr int kNsQueues = 8;    // one work queue per XCD
constexpr int kXcdCus = 32;     // CUs per XCD

// Matrix k owns items [cum[k], cum[k + 1]) of the kind, queue q the range [qlo[q], qlo[q + 1]).
struct NsItems {
  int cum[kNsMaxMats + 1];
  int qlo[kNsQueues + 1];
};

// One matrix: items per phase (P0, P1 or P2, P3) and its estimated work.
struct NsLoad {
  long n0, nt, n3, work;
};

struct NsPlan {
  NsItems i0, it, i3;
  int order[kNsMaxMats];  // the launch's k-th matrix is the given list's order[k]
  int nq;
};

// pinned: one queue per XCD, each matrix on the least loaded one (largest estimated work first, ties to the
// lower index), the list ordered by queue so that a queue's items are a contiguous range. Otherwise one
// device-wide queue. False if a queue's tickets could pass 31 bits.
inline bool ns_place(const NsLoad* m, int n, int nsteps, bool pinned, NsPlan& p) {
  p = NsPlan{};
  p.nq = pinned ? kNsQueues : 1;
  int qof[kNsMaxMats] = {}, first[kNsQueues + 1] = {};
  if (pinned) {
    int by[kNsMaxMats];
    for (int k = 0; k < n; k++) by[k] = k;
    for (int a = 1; a < n; a++)  // stable insertion sort by work, descending
      for (int b = a; b > 0 && m[by[b]].work > m[by[b - 1]].work; b--) std::swap(by[b], by[b - 1]);
    long load[kNsQueues] = {};
    for (int a = 0; a < n; a++) {
      int best = 0;
      for (int q = 1; q < p.nq; q++)
        if (load[q] < load[best]) best = q;
      qof[by[a]] = best;
      load[best] += m[by[a]].work;
    }
  }
  int k2 = 0;
  for (int q = 0; q < p.nq; q++) {
    first[q] = k2;
    for (int k = 0; k < n; k++)
      if (qof[k] == q) p.order[k2++] = k;
  }
  first[p.nq] = k2;
  long c0 = 0, ct = 0, c3 = 0;
  for (int k = 0; k < n; k++) {
    const NsLoad& l = m[p.order[k]];
    c0 += l.n0;
    ct += l.nt;
    c3 += l.n3;
    if (c0 + (long)nsteps * (2 * ct + c3) >= (1L << 31)) return false;
    p.i0.cum[k + 1] = (int)c0;
    p.it.cum[k + 1] = (int)ct;
    p.i3.cum[k + 1] = (int)c3;
  }
  for (int q = 0; q <= p.nq; q++) {
    p.i0.qlo[q] = p.i0.cum[first[q]];
    p.it.qlo[q] = p.it.cum[first[q]];
    p.i3.qlo[q] = p.i3.cum[first[q]];
  }
  return true;
}

}  // namespace ph
