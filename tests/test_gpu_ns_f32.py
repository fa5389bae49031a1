"""fp32 Newton-Schulz: the batched launches against the f64 iteration, at the edges of their 32x32 tiles and
16-wide k chunks, tall and wide, and at the last shape they take and the first that the GEMM chain takes."""
import numpy as np
import pytest
import torch

import oracle_lib as O
from pufferlean_amd import device as D
from pufferlean_amd import rng

pytestmark = pytest.mark.gpu


def ns64(x, coeffs, eps=1e-7):
    y = x.T if x.shape[0] > x.shape[1] else x
    y = y / (np.linalg.norm(y) + eps)
    for a, b, c in coeffs:
        g = y @ y.T
        y = a * y + (b * g + c * (g @ g)) @ y
    return y.T if x.shape[0] > x.shape[1] else y


SHAPES = [(1, 1), (1, 33), (33, 1), (5, 96), (16, 16), (31, 32), (32, 31), (33, 65), (65, 129), (96, 40), (288, 96),
          (128, 512), (200, 129), (127, 500), (2048, 17), (20, 2049)]
# the tier's bar: 5 steps grow a rounding of 6e-8 by up to a^5 ~ 480, and a tile sums up to 2048 products
TOL = 1e-4


@pytest.mark.parametrize("shape", SHAPES)
def test_ns_f32_vs_f64(gpu, shape):
    x0 = rng.normal(0x500 + shape[0] + 3 * shape[1], shape[0] * shape[1], 0.0, 0.02).reshape(shape).astype(np.float32)
    x = torch.from_numpy(x0).cuda()
    D.newton_schulz(x, coeffs=O.REF_COEFFS, math="f32")
    ref = ns64(x0.astype(np.float64), O.REF_COEFFS)
    assert np.linalg.norm(x.cpu().numpy() - ref) <= TOL * np.linalg.norm(ref)


def test_ns_f32_batch_equals_single_calls(gpu):
    """More matrices than one launch holds, an empty one and one for the GEMM chain among them (its extents on the
    vector alignment, where the chain's products on a lane and on the caller's stream are the same kernels)."""
    shapes = SHAPES[:-1] + [(20, 2052), (0, 4), (64, 64), (70, 30)]
    mats = [rng.normal(0x600 + i, r * c, 0.0, 0.02).reshape(r, c).astype(np.float32) for i, (r, c) in enumerate(shapes)]
    batch = [torch.from_numpy(m).cuda() for m in mats]
    D.newton_schulz_batch(batch, coeffs=O.REF_COEFFS, math="f32")
    for m, b in zip(mats, batch):
        one = torch.from_numpy(m).cuda()
        D.newton_schulz(one, coeffs=O.REF_COEFFS, math="f32")
        assert torch.equal(one, b), m.shape


@pytest.mark.parametrize("shape", [(1023, 1024), (1024, 1024)])
def test_ns_f32_large_alone_and_in_a_batch(gpu, shape):
    """The last shape of the launches and the first of the chain near 1024: the f64 iteration's result, and in a batch of
    four the same bits as alone."""
    x0 = rng.normal(0x700 + shape[0], shape[0] * shape[1], 0.0, 0.02).reshape(shape).astype(np.float32)
    one = torch.from_numpy(x0).cuda()
    D.newton_schulz(one, coeffs=O.REF_COEFFS, math="f32")
    ref = ns64(x0.astype(np.float64), O.REF_COEFFS)
    assert np.linalg.norm(one.cpu().numpy() - ref) <= TOL * np.linalg.norm(ref)
    batch = [torch.from_numpy(x0).cuda() for _ in range(4)] + [torch.from_numpy(x0[:60, :90].copy()).cuda()]
    D.newton_schulz_batch(batch, coeffs=O.REF_COEFFS, math="f32")
    for b in batch[:4]:
        assert torch.equal(b, one)
