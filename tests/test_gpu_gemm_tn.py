"""TN products (weight gradients) whose reduction length is no multiple of the vector width: they run in
place, by whole k-rows, on 64x64 and 128x128 split-K tiles, with a fold of few and of many splits.

The fp32 result is compared with the f64 product of the operands as the kernel reads them: sums of K products
in fp32, each partial within K 2^-24 relative of the sum of magnitudes; 1e-5 (relative Frobenius) is the
library's fp32 bar and above the 4e-7 that random signs give."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture
def D():
    from pufferlean_amd import device
    return device


@pytest.mark.parametrize("K", [1, 7, 63, 4097, 6699, 33001])
@pytest.mark.parametrize("M,N", [(8, 8), (32, 96), (136, 40), (288, 96), (64, 520)])
@pytest.mark.parametrize("dt,math", [("f32", "f32"), ("f32", "bf16"), ("bf16", "bf16")])
def test_tn_any_k(D, M, N, K, dt, math):
    g = torch.Generator(device="cuda").manual_seed(K * 1000 + M + N)
    t = torch.bfloat16 if dt == "bf16" else torch.float32
    # NaN rows past the end: a read beyond K would poison the sums
    a = torch.full((K + 8, M), float("nan"), device="cuda", dtype=t)
    b = torch.full((K + 8, N), float("nan"), device="cuda", dtype=t)
    a[:K] = torch.randn(K, M, generator=g, device="cuda").to(t)
    b[:K] = torch.randn(K, N, generator=g, device="cuda").to(t)
    out = D.gemm(a[:K], b[:K], trans_a=True, math=math)
    r = (lambda x: x.bfloat16().double()) if math == "bf16" else (lambda x: x.double())
    ref = r(a[:K]).t() @ r(b[:K])
    err = ((out.double() - ref).norm() / ref.norm()).item()
    print(f"TN {M}x{N}x{K} {dt}/{math}: {err:.2e}", flush=True)
    assert err < 1e-5


@pytest.mark.parametrize("B,T", [(7, 13), (45, 31)])
def test_mingru_gradient_odd_rows(D, B, T):
    """The head's weight gradient runs on an update lane: an odd row count T*B takes the same kernels as an
    even one (the gradient of a batch is the sum of its segments' gradients)."""
    g = torch.Generator(device="cuda").manual_seed(B)
    Dm, H, L, A = 16, 64, 1, 5
    kw = dict(precision="f32")
    cfg = D.MinGRUConfig(B, T, Dm, H, L, A, **kw)
    one = D.MinGRUConfig(1, T, Dm, H, L, A, **kw)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda")
    p = rn(cfg.P) * 0.1
    obs, act = rn(T, B, Dm), torch.randint(0, A, (T, B), generator=g, device="cuda", dtype=torch.int32)
    cols = [rn(T, B) for _ in range(4)]
    cols[2] = cols[2] * 0.1 - 1.6
    done = (torch.rand(T, B, generator=g, device="cuda") < 0.1).float()
    G, _, _ = D.mingru_ppo_grad(cfg, p, obs, act, *cols, done)
    ref = torch.zeros(cfg.P, device="cuda", dtype=torch.float64)
    for b in range(B):
        c = lambda x: x[:, b:b + 1].contiguous()
        Gb, _, _ = D.mingru_ppo_grad(one, p, c(obs), c(act), *[c(x) for x in cols], c(done))
        ref += Gb.double()
    err = ((G.double() - ref).norm() / ref.norm()).item()
    print(f"mingru odd rows B={B} T={T}: {err:.2e}", flush=True)
    assert err < 1e-5


@pytest.mark.parametrize("M,N,K,ta,tb", [(64, 8256, 4096, 1, 0), (64, 8256, 4100, 0, 1), (9000, 32, 4097, 1, 0), (9000, 30, 4096, 0, 1),
                                         (512, 64, 16384, 1, 0), (512, 64, 16392, 1, 0), (64, 130, 70001, 1, 0), (48, 100, 5003, 0, 0)])
@pytest.mark.parametrize("math", ["f32", "bf16"])
def test_narrow_outputs(D, M, N, K, ta, tb, math):
    """Long reductions with an output at most 64 wide or tall, on both sides of the rule for 64x64 split tiles. The bar as
    above; rows past the end hold NaN."""
    g = torch.Generator(device="cuda").manual_seed(M + N + K)

    def operand(r, c):
        x = torch.full((r + 4, c), float("nan"), device="cuda")
        x[:r] = torch.randn(r, c, generator=g, device="cuda")
        return x[:r]
    a = operand(*((K, M) if ta else (M, K)))
    b = operand(*((N, K) if tb else (K, N)))
    out = D.gemm(a, b, trans_a=bool(ta), trans_b=bool(tb), math=math)
    r = (lambda x: x.bfloat16().double()) if math == "bf16" else (lambda x: x.double())
    ref = (r(a).t() if ta else r(a)) @ (r(b).t() if tb else r(b))
    err = ((out.double() - ref).norm() / ref.norm()).item()
    print(f"{M}x{N}x{K} ta={ta} tb={tb} {math}: {err:.2e}", flush=True)
    assert err < 1e-5


@pytest.mark.parametrize("M,N,splits", [(64, 64, 63), (64, 64, 64), (64, 64, 255), (64, 64, 256), (72, 64, 256), (256, 256, 65),
                                        (264, 256, 65), (8, 8, 300)])
@pytest.mark.parametrize("cdt", [torch.float32, torch.bfloat16])
def test_fold_forms(D, M, N, splits, cdt):
    """One, four and sixteen threads per element of the fold, around the lines between them, with whole and ragged ranges
    of splits (64 of k each, the last shorter). bf16 outputs are the rounded sums: 2^-8 per element."""
    K = 64 * splits - 13
    g = torch.Generator(device="cuda").manual_seed(M + splits)
    a, b = (torch.randn(K, n, generator=g, device="cuda") for n in (M, N))
    out = D.gemm(a, b, trans_a=True, math="f32", splits=splits, out_dtype=cdt)
    ref = a.double().t() @ b.double()
    err = ((out.double() - ref).norm() / ref.norm()).item()
    assert err < (1e-5 if cdt == torch.float32 else 2 ** -8)


@pytest.mark.parametrize("M,N,K", [(136, 200, 4097), (128, 256, 5001), (512, 512, 131079), (264, 136, 262147), (8192, 2048, 77)],
                         ids=["128x256", "128x256-ragged-splits", "256x256-dma", "256x256-dma-ragged-tile", "256x128"])
def test_tn_any_k_large_tiles(D, M, N, K):
    """The bf16 kernels of the large weight gradients with a reduction that ends inside a k-tile: 128x256 splits, the
    load-to-LDS kernel at 256x256 and the unsplit 256x128 tiles. Rows past the end hold NaN."""
    g = torch.Generator(device="cuda").manual_seed(K)
    a, b = (torch.full((K + 40, n), float("nan"), device="cuda", dtype=torch.bfloat16) for n in (M, N))
    for x in (a, b):
        x[:K] = torch.randn(K, x.shape[1], generator=g, device="cuda").bfloat16()
    print(f"TN {M}x{N}x{K}", flush=True)
    out = D.gemm(a[:K], b[:K], trans_a=True)
    ref = torch.zeros(M, N, device="cuda", dtype=torch.float64)
    for k0 in range(0, K, 32768):
        ref += a[k0:min(K, k0 + 32768)].double().t() @ b[k0:min(K, k0 + 32768)].double()
    assert ((out.double() - ref).norm() / ref.norm()).item() < 1e-5


@pytest.mark.parametrize("M,N,K", [(136, 40, 4099), (40, 64, 9001), (304, 96, 999), (256, 256, 4101)])
def test_tn_any_k_split_bf16(D, M, N, K):
    """Split-bf16 products of a ragged reduction. Each operand is held to 2^-17 of its value and the product of the two low
    halves (2^-18) is dropped: 2.5 x 2^-17 and the fp32 sums' 1e-5."""
    from pufferlean_amd import _lib as L
    g = torch.Generator(device="cuda").manual_seed(K)
    a, b = (torch.full((K + 8, n), float("nan"), device="cuda") for n in (M, N))
    for x in (a, b):
        x[:K] = torch.randn(K, x.shape[1], generator=g, device="cuda")
    out = torch.empty(M, N, device="cuda")
    p = lambda x: D._p(x)
    L.call("ph_gemm", 1, 0, M, N, K, L.PH_F32, p(a), M, L.PH_F32, p(b), N, L.PH_F32, p(out), N, L.PH_MATH_BF16X3,
           L.PH_EPI_NONE, None, None, 0, 1.0, 0.0, None, 0, 0, 0, D._stream())
    ref = a[:K].double().t() @ b[:K].double()
    assert ((out.double() - ref).norm() / ref.norm()).item() < 2.5 * 2 ** -17 + 1e-5
