"""The rules that choose a kernel's form (csrc/routes.hpp) on the host, at sizes where the other form measured slower."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = r"""
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include "routes.hpp"
using namespace ph;
int main(int argc, char** argv) {
  long a[8] = {};
  for (int i = 2; i < argc && i < 10; i++) a[i - 2] = std::atol(argv[i]);
  long r = -1;
  if (!std::strcmp(argv[1], "gemm_small_splits")) r = gemm_small_splits(a[0], a[1], a[2], a[3], a[4], a[5]);
  if (!std::strcmp(argv[1], "fold_threads")) r = fold_threads((int)a[0], a[1]);
  if (!std::strcmp(argv[1], "sample_registers")) r = sample_registers(a[0]);
  if (!std::strcmp(argv[1], "vtrace_tiled")) r = vtrace_tiled(a[0], a[1], a[2], a[3]);
  if (!std::strcmp(argv[1], "gather_tiled")) r = gather_tiled(a[0], a[1]);
  if (!std::strcmp(argv[1], "seg_l1_tiled")) r = seg_l1_tiled(a[0], a[1], a[2], a[3]);
  if (!std::strcmp(argv[1], "prio_one_block")) r = prio_one_block(a[0], a[1]);
  if (!std::strcmp(argv[1], "iterate_tiled")) r = iterate_tiled(a[0], a[1], a[2]);
  if (!std::strcmp(argv[1], "gather_folds")) r = gather_folds(a[0]);
  if (!std::strcmp(argv[1], "rollout_form")) r = rollout_form(a[0], a[1], a[2]);
  if (!std::strcmp(argv[1], "ns_f32_fits")) r = ns_f32_fits((int)a[0], (int)a[1]);
  std::printf("%ld\n", r);
  return 0;
}
"""


@pytest.fixture(scope="module")
def route(tmp_path_factory):
    d = tmp_path_factory.mktemp("routes")
    (d / "drv.cpp").write_text(DRIVER)
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "pufferlean_amd", "csrc"),
                    "-o", str(d / "drv"), str(d / "drv.cpp")], check=True)

    def call(name, *args):
        out = subprocess.run([str(d / "drv"), name] + [str(int(x)) for x in args], capture_output=True, text=True, check=True)
        return int(out.stdout)
    return call


# (fp32 math, trans_b, M, N, K) of products of fp32 operands, and whether 64x64 splits are the faster form
GEMM = [
    (0, 0, 64, 8256, 4096, 0), (0, 0, 64, 8256, 32768, 0), (0, 1, 64, 8256, 16384, 0), (0, 0, 16, 9000, 8192, 0),
    (0, 0, 8256, 64, 8192, 0), (0, 1, 9000, 32, 8192, 0), (0, 0, 512, 64, 32768, 0), (0, 0, 512, 32, 262144, 0),
    (0, 0, 2048, 32, 32768, 0), (0, 0, 64, 256, 65536, 0), (0, 0, 64, 64, 65536, 1), (0, 0, 128, 64, 262144, 1),
    (0, 0, 64, 1024, 8192, 1), (0, 0, 64, 4096, 8192, 1), (0, 1, 64, 5120, 8192, 0),
    (0, 0, 512, 32, 8192, 1), (0, 0, 65, 65, 65536, 0), (1, 1, 64, 8256, 16384, 0),
    (1, 1, 9000, 32, 8192, 0), (1, 0, 64, 8256, 16384, 1), (1, 1, 64, 4096, 8192, 1), (1, 0, 512, 64, 262144, 1),
    (1, 0, 288, 96, 6699, 1), (1, 0, 512, 512, 16384, 0), (1, 0, 128, 256, 65536, 0),
]


@pytest.mark.parametrize("f32,tb,M,N,K,small", GEMM)
def test_gemm_small_splits(route, f32, tb, M, N, K, small):
    assert route("gemm_small_splits", f32, 1, tb, M, N, K) == small
    assert route("gemm_small_splits", 0, 0, tb, M, N, K) == 0  # bf16 operands never


@pytest.mark.parametrize("splits,MN,threads", [(128, 128 * 128, 4), (128, 64 * 512, 4), (256, 256 * 128, 4), (64, 256 * 256, 4),
                                               (32, 64 * 64, 1), (32, 512 * 64, 1), (16, 512 * 512, 1), (64, 512 * 256, 1),
                                               (512, 8 * 8, 16), (512, 128 * 64, 4)])
def test_fold_threads(route, splits, MN, threads):
    assert route("fold_threads", splits, MN) == threads


@pytest.mark.parametrize("A,regs", [(1, 0), (2, 4), (4, 4), (5, 8), (8, 8), (9, 16), (16, 16), (17, 32), (32, 32), (33, 0)])
def test_sample_registers(route, A, regs):
    assert route("sample_registers", A) == regs


# (f64, time-major, B, T) and whether the tiles are the faster form
VTRACE = [(0, 1, 4096, 1, 0), (0, 1, 4096, 4, 0), (0, 1, 4096, 8, 1), (0, 1, 16384, 8, 0), (0, 1, 16384, 16, 0),
          (0, 1, 16384, 64, 1), (0, 1, 32767, 8, 0), (0, 1, 32767, 64, 1), (0, 1, 32767, 72, 0), (0, 1, 32768, 64, 0),
          (1, 1, 4096, 4, 0), (1, 1, 8192, 8, 0), (1, 1, 4096, 64, 1), (1, 1, 16384, 12, 0), (1, 1, 16384, 64, 1),
          (1, 1, 24576, 16, 0), (1, 1, 24576, 65, 0), (1, 1, 24576, 128, 1), (1, 1, 32767, 65, 0), (0, 0, 4096, 1, 0),
          (0, 0, 4096, 4, 1), (0, 0, 16384, 4, 0), (0, 0, 16384, 8, 1), (0, 0, 65536, 1, 0), (0, 0, 65536, 8, 0),
          (0, 0, 65536, 64, 1), (1, 0, 256, 4, 0), (1, 0, 4096, 8, 1), (1, 0, 32767, 8, 0), (1, 0, 65536, 2, 0),
          (1, 0, 65536, 64, 1), (0, 0, 93, 5, 0), (0, 0, 129, 5, 1), (0, 0, 93, 8, 1), (1, 1, 188, 11, 1), (1, 1, 8192, 11, 0)]


@pytest.mark.parametrize("f64,tm,B,T,tiled", VTRACE)
def test_vtrace_tiled(route, f64, tm, B, T, tiled):
    assert route("vtrace_tiled", f64, tm, B, T) == tiled


@pytest.mark.parametrize("f64,N,T,tiled", [(0, 65536, 16, 0), (0, 4096, 24, 0), (0, 4096, 63, 0), (0, 4096, 64, 1), (0, 16, 4096, 0),
                                           (0, 127, 2048, 0), (0, 128, 2048, 1), (1, 65536, 17, 0), (1, 4096, 24, 0),
                                           (1, 4096, 32, 1), (1, 16, 4096, 1)])
def test_seg_l1_tiled(route, f64, N, T, tiled):
    assert route("seg_l1_tiled", f64, 0, N, T) == tiled
    assert route("seg_l1_tiled", f64, 1, N, T) == 0


@pytest.mark.parametrize("T,tiled", [(15, 0), (16, 1), (4096, 1)])
def test_gather_tiled(route, T, tiled):
    assert route("gather_tiled", 0, T) == tiled and route("gather_tiled", 1, T) == 0


@pytest.mark.parametrize("N,draws,one", [(1, 1, 1), (64, 64, 1), (1024, 1024, 1), (2048, 1024, 1), (2049, 64, 0), (64, 1025, 0), (1024, 2048, 0),
                                         (4096, 4096, 0)])
def test_prio_one_block(route, N, draws, one):
    assert route("prio_one_block", N, draws) == one


@pytest.mark.parametrize("draws,T,tiled", [(64, 15, 0), (64, 16, 1), (4096, 16, 1), (4097, 47, 0), (4097, 48, 1), (8192, 16, 0),
                                           (8192, 32, 0), (8192, 64, 1), (16, 1024, 1), (4096, 256, 1), (8193, 256, 0)])
def test_iterate_tiled(route, draws, T, tiled):
    assert route("iterate_tiled", 0, draws, T) == tiled and route("iterate_tiled", 1, draws, T) == 0


@pytest.mark.parametrize("blocks,folds", [(1, 1), (1024, 1), (1025, 0), (2048, 0)])
def test_gather_folds(route, blocks, folds):
    assert route("gather_folds", blocks) == folds


# (bf16, rows, units) and the faster form: 0 the GEMM chain, 1, 2 and 3 blocks of 32, 128 and 256 rows
ROLLOUT = [(1, 48, 128, 1), (1, 2048, 128, 1), (1, 16384, 128, 3), (1, 4096, 256, 2), (1, 6000, 256, 3), (1, 512, 512, 1),
           (1, 700, 512, 2), (1, 2048, 512, 2), (1, 2600, 512, 3), (1, 4096, 512, 3), (1, 1500, 384, 2), (1, 3300, 384, 3),
           (1, 1024, 640, 2), (1, 300, 1024, 2), (1, 2600, 768, 2), (1, 200, 1280, 2), (1, 48, 2048, 0), (1, 200, 2048, 2),
           (1, 48, 4096, 0), (0, 48, 128, 1), (0, 8192, 128, 2), (0, 2048, 384, 1), (0, 1300, 512, 1), (0, 2048, 512, 2),
           (0, 4096, 512, 2), (0, 6000, 256, 1), (0, 4096, 640, 0), (0, 7072, 328, 0), (0, 2600, 768, 2), (0, 3300, 768, 0), (0, 48, 896, 1),
           (0, 300, 896, 0), (0, 700, 896, 0), (0, 1, 1024, 0), (0, 1024, 1024, 2), (0, 2600, 1024, 0), (0, 48, 2048, 0),
           (0, 2048, 1280, 0), (0, 1024, 2048, 2), (0, 1024, 2056, 0)]


@pytest.mark.parametrize("bf,N,H,form", ROLLOUT)
def test_rollout_form(route, bf, N, H, form):
    assert route("rollout_form", bf, N, H) == form


@pytest.mark.parametrize("rows,cols,fits", [(512, 512, 1), (1023, 1023, 1), (2048, 1023, 1), (2048, 64, 1), (1023, 1100, 1),
                                            (1024, 1024, 0), (1100, 1151, 0), (1024, 1152, 1), (1152, 1024, 1),
                                            (1536, 1536, 1), (2048, 1536, 1), (2048, 1537, 0), (2049, 8, 0), (8, 2049, 0)])
def test_ns_f32_fits(route, rows, cols, fits):
    assert route("ns_f32_fits", rows, cols) == fits
