"""Placement of a fused Newton-Schulz launch (csrc/ns_plan.hpp) on the host: the launch drains when the queues' blocks
start late, one at a time and in any order of the queues."""
import os
import subprocess
import textwrap

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# One block per queue, the queues served one after the other: a block takes its queue's tickets in order and may
# run an item only when every item of the matrix's earlier phases is done. No block of a later queue has
# started yet, so an item that needs one would wait for ever.
DRIVER = textwrap.dedent(r"""
    #include <cstdio>
    #include <cstdlib>
    #include <cstring>
    #include "ns_plan.hpp"
    using namespace ph;
    static int owner(const int* cum, int n, int i) { int k = 0; while (k + 1 < n && i >= cum[k + 1]) k++; return k; }
    int main(int argc, char** argv) {  // pinned, then rows cols ...
      const bool pinned = std::atoi(argv[1]) != 0;
      const int steps = 5, n = (argc - 2) / 2;
      NsLoad m[kNsMaxMats] = {};
      for (int k = 0; k < n; k++) {
        const int r = std::atoi(argv[2 + 2 * k]), c = std::atoi(argv[3 + 2 * k]);
        const long tm = ((r < c ? r : c) + 63) / 64, tw = ((r < c ? c : r) + 63) / 64, nt = tm * (tm + 1) / 2;
        m[k] = NsLoad{tm * tw, nt, tm * tw, tm * tw + steps * (nt * tw + 3 * nt * tm + 3 * tm * tw * tm)};
      }
      NsPlan p;
      if (!ns_place(m, n, steps, pinned, p)) return 2;
      int seen[kNsMaxMats] = {};
      for (int k = 0; k < n; k++) seen[p.order[k]]++;
      for (int k = 0; k < n; k++) if (seen[k] != 1) { std::printf("matrix %d listed %d times\n", k, seen[k]); return 1; }
      for (int first = 0; first < p.nq; first++) {
        long done[kNsMaxMats] = {};
        for (int v = 0; v < p.nq; v++) {
          const int q = (first + 5 * v) % p.nq;  // every queue once (p.nq is 1 or 8)
          for (int ph = 0; ph <= 3 * steps; ph++) {
            const int kind = ph == 0 ? 0 : (ph - 1) % 3 + 1;
            const NsItems& it = kind == 0 ? p.i0 : kind == 3 ? p.i3 : p.it;
            for (int i = it.qlo[q]; i < it.qlo[q + 1]; i++) {
              const int k = owner(it.cum, n, i);
              const NsLoad& l = m[p.order[k]];
              const int s = ph == 0 ? 0 : (ph - 1) / 3;
              const long need = kind == 0 ? 0 : l.n0 + s * (2 * l.nt + l.n3) + (kind - 1) * l.nt;
              if (done[k] < need) { std::printf("queue %d phase %d matrix %d waits for another queue\n", q, ph, k); return 1; }
              done[k]++;
            }
          }
        }
        for (int k = 0; k < n; k++) {
          const NsLoad& l = m[p.order[k]];
          if (done[k] != l.n0 + steps * (2 * l.nt + l.n3)) { std::printf("matrix %d ran %ld items\n", k, done[k]); return 1; }
        }
      }
      std::printf("ok\n");
      return 0;
    }
""")


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    d = tmp_path_factory.mktemp("ns_plan")
    (d / "drv.cpp").write_text(DRIVER)
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "pufferlean_amd", "csrc"),
                    "-o", str(d / "drv"), str(d / "drv.cpp")], check=True)
    return str(d / "drv")


SHAPES = [[(512, 512)], [(1536, 512)], [(768, 768)], [(512, 512)] * 4, [(700, 330), (40, 900)], [(512, 512)] * 6,
          [(1536, 512), (512, 128), (16, 512), (1, 512)], [(64, 64)] * 14 + [(256, 256), (3, 128)], [(128, 4)]]


@pytest.mark.parametrize("pinned", [0, 1])
@pytest.mark.parametrize("shapes", SHAPES, ids=["+".join("%dx%d" % s for s in sh[:3]) + "-%d" % len(sh) for sh in SHAPES])
def test_drains_with_late_queues(driver, shapes, pinned):
    r = subprocess.run([driver, str(pinned)] + [str(x) for s in shapes for x in s], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout
