"""Head gradients through the LDS tile: row counts around a block's 256 rows, odd and even row widths, one to eight
heads, the largest around the lines between the column passes, packed rows (moved as one run of floats), strided
rows and rows off the 16-byte alignment."""
import numpy as np
import pytest
import torch

import oracle_lib as O
from pufferlean_amd import device as D
from pufferlean_amd import rng

pytestmark = pytest.mark.gpu


def cu(x, dt=torch.float32):
    return torch.from_numpy(np.ascontiguousarray(x)).to("cuda", dt)


def rows(x, layout):
    """x's rows packed, at a wider stride, or packed from a base one float past a 16-byte boundary."""
    n, w = x.shape
    if layout == "packed":
        return x.clone()
    if layout == "strided":
        buf = torch.full((n, w + 3), 7.0, device="cuda")
        buf[:, :w] = x
        return buf[:, :w]
    buf = torch.empty(n * w + 1, device="cuda")
    v = buf[1:].view(n, w)
    v.copy_(x)
    return v


f32 = lambda x: x.astype(np.float32).astype(np.float64)
LAYOUTS = ["packed", "strided", "offset"]


@pytest.mark.parametrize("N", [1, 63, 255, 256, 257, 1001])
@pytest.mark.parametrize("sizes", [[1], [2], [9, 5], [3, 3, 4, 1], [31], [1, 2, 3, 4, 5, 6, 7, 3], [12, 7, 3],
                                   [13, 2], [16, 15], [17, 1], [24, 3], [25]])
def test_md_tile(gpu, N, sizes):
    K, W = len(sizes), sum(sizes)
    out = f32(rng.normal(0xB01 + N, N * (W + 1)).reshape(N, W + 1) * 2.0)
    acts = np.stack([rng.randint(0xB02 + h, N, s) for h, s in enumerate(sizes)], axis=1)
    adv, ret, ov = (f32(rng.normal(0xB06 + i, N)) for i in range(3))
    _, nlp0, _ = O.ppo_grad_md(out, acts, adv, ret, np.zeros(N), ov, sizes)
    old = f32(nlp0 + rng.normal(0xB09, N, 0.0, 0.3))
    ref, rlp, rv = O.ppo_grad_md(out, acts, adv, ret, old, ov, sizes, vfclip=0.2)
    got = {}
    for lay in LAYOUTS:
        o, d = rows(cu(out), lay), rows(torch.zeros(N, W + 1, device="cuda"), lay)
        nlp, nv = torch.empty(N, device="cuda"), torch.empty(N, device="cuda")
        losses = torch.zeros(7, device="cuda", dtype=torch.float64)
        ins = cu(acts, torch.int32), cu(adv), cu(ret), cu(old), cu(ov)
        D.ppo_grad_md(o, *ins, head_sizes=sizes, vf_clip=0.2, dout=d, newlp=nlp, newval=nv, losses=losses)
        got[lay] = [x.cpu().numpy() for x in (d, nlp, nv, losses)]
        if lay == "strided":  # nothing past the row width is written
            assert torch.all(d.as_strided((N, 3), (W + 4, 1), W + 1) == 7.0)
    g, nlp, nv, losses = got["packed"]
    assert np.linalg.norm(g - ref) <= 1e-5 * np.linalg.norm(ref)  # the fp32 heads' bar
    np.testing.assert_allclose(nlp, rlp, rtol=1e-5, atol=1e-5)
    assert np.array_equal(nv.astype(np.float64), rv)
    for lay in LAYOUTS[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(got["packed"], got[lay])), lay


@pytest.mark.parametrize("N", [1, 256, 257, 1001])
@pytest.mark.parametrize("dim", [1, 2, 4, 5, 8, 15])
def test_cont_tile(gpu, N, dim):
    w = 2 * dim + 1
    out = rng.normal(0xB11 + N, N * w).reshape(N, w)
    out[:, dim:2 * dim] *= 0.5
    out = f32(out)
    acts = f32(out[:, :dim] + rng.normal(0xB12, N * dim).reshape(N, dim) * 0.5)
    adv, ret, ov = (f32(rng.normal(0xB16 + i, N)) for i in range(3))
    _, nlp0, _ = O.ppo_grad_cont(out, acts, adv, ret, np.zeros(N), ov, dim)
    old = f32(nlp0 + rng.normal(0xB19, N, 0.0, 0.1))
    ref, rlp, _ = O.ppo_grad_cont(out, acts, adv, ret, old, ov, dim, vfclip=0.2)
    got = {}
    for lay in LAYOUTS:
        o, d = rows(cu(out), lay), rows(torch.zeros(N, w, device="cuda"), lay)
        nlp, nv = torch.empty(N, device="cuda"), torch.empty(N, device="cuda")
        losses = torch.zeros(7, device="cuda", dtype=torch.float64)
        ins = cu(acts), cu(adv), cu(ret), cu(old), cu(ov)
        D.ppo_grad_cont(o, *ins, dim=dim, vf_clip=0.2, dout=d, newlp=nlp, newval=nv, losses=losses)
        got[lay] = [x.cpu().numpy() for x in (d, nlp, nv, losses)]
    g, nlp = got["packed"][:2]
    assert np.linalg.norm(g - ref) <= 1e-5 * np.linalg.norm(ref)
    np.testing.assert_allclose(nlp, rlp, rtol=1e-5, atol=1e-5)
    for lay in LAYOUTS[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(got["packed"], got[lay])), lay
