"""The rollout step's fused layers and head: tile remainders of rows, units and k, the rule between its three
layer kernels, and the sampler's register forms.

fp32: each product sums H terms in fp32 (another order than the f64 reference): 1e-5 relative, the library's
fp32 bar. bf16: operands rounded to 8 bits, 2e-2 over a step of up to three layers, as the rollout tests state."""
from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture
def D():
    from pufferlean_amd import device
    return device


def reference(p, obs, state, D_, H, L, A):
    p, obs, state = p.double(), obs.double(), state.double()
    off = 0

    def take(r, c):
        nonlocal off
        v = p[off:off + r * c].view(r, c)
        off += r * c
        return v
    x = obs @ take(H, D_).t() + take(1, H)
    new = []
    for l in range(L):
        hid, gate, proj = (x @ take(3 * H, H).t()).chunk(3, 1)
        z, hg = torch.sigmoid(gate), torch.sigmoid(proj)
        o = (1 - z) * state[:, l] + z * torch.where(hid >= 0, hid + 0.5, torch.sigmoid(hid))
        new.append(o)
        x = hg * o + (1 - hg) * x
    wd, bd, wv, bv = take(A, H), take(1, A), take(1, H), take(1, 1)
    return torch.cat([x @ wd.t() + bd, x @ wv.t() + bv], 1), torch.stack(new, 1)


# 8 and 40: units and k below and past a 32-unit tile; 72: a ragged second k chunk; 7: the unfused path.
# Row counts around the 32, 128 and 256 row tiles and, at H = 512, the rule between them.
@pytest.mark.parametrize("N,H", [(1, 8), (31, 40), (33, 72), (48, 128), (129, 24), (257, 96), (5, 7), (1500, 512),
                                 (1536, 512), (3071, 512), (3100, 512), (2305, 264)])
@pytest.mark.parametrize("A,L", [(1, 1), (6, 2), (31, 3)])
@pytest.mark.parametrize("precision", [0, 1])
def test_step(D, N, H, A, L, precision):
    D_ = 12
    g = torch.Generator(device="cuda").manual_seed(N + H)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda")
    P = H * D_ + H + L * 3 * H * H + A * H + A + H + 1
    p = rn(P) / np.sqrt(H)
    obs, state = rn(N, D_), rn(N, L, H)
    out = torch.full((N, A + 1), float("nan"), device="cuda")
    ref_out, ref_state = reference(p, obs, state, D_, H, L, A)
    guard = torch.full((N + 8, L, H), 7.0, device="cuda")  # rows past N stay untouched
    guard[:N] = state
    print(f"rollout N={N} H={H} A={A} L={L} precision={precision}", flush=True)
    D.mingru_rollout_step(p, obs, guard[:N], out, D=D_, H=H, L_layers=L, A=A, precision=precision)
    tol = 1e-5 if precision else 2e-2
    assert ((out.double() - ref_out).norm() / ref_out.norm()).item() < tol
    assert ((guard[:N].double() - ref_state).norm() / ref_state.norm()).item() < tol
    assert bool((guard[N:] == 7.0).all())


# both sides of the lines between the forms: 700 and 2600 rows of 512 units, few rows of 1280 and more, fp32 past 768
# units and where the chain's tiles fill their rounds
@pytest.mark.parametrize("N,H", [(700, 512), (2600, 512), (33, 1288), (129, 1288), (3, 2056), (256, 776), (257, 776), (40, 904),
                                 (300, 320), (3300, 768)])
@pytest.mark.parametrize("precision", [0, 1])
def test_step_forms(D, N, H, precision):
    test_step(D, N, H, 6, 1, precision)


@pytest.mark.parametrize("dt", [torch.float32, torch.float64])
@pytest.mark.parametrize("A", [1, 2, 4, 5, 8, 9, 15, 16, 17, 32, 33])
def test_sampler_widths(D, A, dt):
    """Register forms (up to 4, 8, 16 and 32 logits) and the wide form against numpy's softmax and inverse CDF; a draw
    within 1e-5 (f32) or 1e-12 (f64) of a cumulative boundary may take the neighbour."""
    from pufferlean_amd import rng
    N = 777
    Y = torch.randn(N, A + 2, generator=torch.Generator().manual_seed(A), dtype=torch.float64).to(dt)
    Y[5, :A] = -float("inf")
    Y[5, A - 1] = 3.0  # all the mass on the last action
    act, lp, val = D.sample_actions(Y.cuda()[:, :A + 1], A, rng_state=0x1234)
    p = torch.softmax(Y[:, :A].double(), 1).numpy()
    cum = np.cumsum(p, 1)
    u = rng.uniform01(rng.words(0x1234, N))
    ref = np.minimum((cum <= u[:, None]).sum(1), A - 1)
    got = act.cpu().numpy()
    eps = 1e-5 if dt == torch.float32 else 1e-12
    for n in np.nonzero(got != ref)[0]:
        assert abs(cum[n, min(got[n], ref[n])] - u[n]) < eps
    np.testing.assert_allclose(lp.cpu().numpy(), np.log(p[np.arange(N), got]), rtol=0, atol=1e-5 if dt == torch.float32 else 1e-12)
    assert torch.equal(val.cpu(), Y[:, A])
