"""Segment-major replay columns through the 16-segment x 64-step tiles: steps and draws around the tile's edges and
the rule's limits, both types, several action components, repeated and invalid draws; and the sampler around the
lines between its three forms."""
import numpy as np
import pytest
import torch

import oracle_lib as O
from pufferlean_amd import device as D
from pufferlean_amd import rng

pytestmark = pytest.mark.gpu

DT = {"f64": (torch.float64, np.float64, 1e-12), "f32": (torch.float32, np.float32, 1e-6)}


def columns(N, T, K, np_dt, dt):
    c = {n: rng.normal(0x701 + i, N * T).reshape(N, T).astype(np_dt) for i, n in enumerate(("adv", "value", "logp"))}
    c["term"] = (rng.randf(0x705, N * T, 0.0, 1.0).reshape(N, T) < 0.2).astype(np_dt)
    c["act"] = rng.randint(0x706, N * T * K, 8).reshape(N, T, K).astype(np_dt)
    return c, {k: torch.from_numpy(v).to("cuda", dt) for k, v in c.items()}


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("N,T,B,K", [(1, 16, 1, 1), (40, 15, 17, 2), (40, 17, 16, 1), (15, 64, 15, 3), (33, 65, 100, 2),
                                     (17, 130, 33, 1), (100, 520, 4096, 1),
                                     (128, 63, 5, 1), (129, 64, 20, 1), (127, 70, 9, 1), (20, 31, 9, 1), (20, 32, 9, 1)])
def test_tiles(gpu, dtype, N, T, B, K):
    dt, np_dt, tol = DT[dtype]
    h, d = columns(N, T, K, np_dt, dt)
    seg = rng.randint(0x710, B, N)
    if B > 8:
        seg[[3, 7]] = [-1, N]
        seg[5] = seg[2] = seg[B - 1]
    ok = (seg >= 0) & (seg < N)
    mp = rng.randf(0x711, B, 0.3, 3.0)
    ratio = torch.ones(N, T, device="cuda", dtype=dt)
    cols = D.ReplayColumns(N, T, **d, ratio=ratio, K=K)
    # sums in the order of the steps, in f64
    l1 = np.zeros(N)
    for t in range(T):
        l1 += np.abs(h["adv"][:, t].astype(np.float64))
    assert np.array_equal(D.seg_l1(cols).cpu().numpy(), l1)
    # gathered columns
    dseg = torch.from_numpy(seg).to("cuda", torch.int32)
    sel = np.where(ok, seg, 0)
    tm = lambda x: np.where(ok, x[sel].T, np.nan)  # [T, B]
    if ok.all():  # an invalid draw's NaN reaches the mean, as in every form
        out = D.mb_gather(cols, dseg, torch.from_numpy(mp).cuda()).cpu().numpy()
        a = tm(h["adv"]).astype(np.float64)
        norm = mp * (a - a.mean()) / (a.std() + 1e-8)
        got = out[K * T * B:].reshape(5, T, B)
        assert np.max(np.abs(got[0] - norm)) <= tol * np.max(np.abs(norm))
    else:
        out = D.mb_gather(cols, dseg, torch.from_numpy(mp).cuda()).cpu().numpy()
        got = out[K * T * B:].reshape(5, T, B)
        assert np.isnan(got[0]).all()
    act = np.where(ok[None, :, None], h["act"][sel].transpose(1, 0, 2), np.nan)
    assert np.array_equal(out[:K * T * B].reshape(T, B, K), act, equal_nan=True)
    for col, ref in ((1, h["adv"] + h["value"]), (2, h["logp"]), (3, h["term"]), (4, h["value"])):
        assert np.array_equal(got[col], tm(ref), equal_nan=True), col
    # the last draw of a segment leaves its values
    newlp, newval = rng.normal(0x720, T * B).astype(np.float32), rng.normal(0x721, T * B).astype(np.float32)
    D.mb_iterate(cols, dseg, torch.from_numpy(newlp).cuda(), torch.from_numpy(newval).cuda())
    ev, er = h["value"].copy(), np.ones((N, T), np_dt)
    for b in range(B):
        if ok[b]:
            ev[seg[b]] = newval.reshape(T, B)[:, b]
            er[seg[b]] = np.exp(newlp.reshape(T, B)[:, b].astype(np.float64) - h["logp"][seg[b]].astype(np.float64))
    assert np.array_equal(d["value"].cpu().numpy(), ev)
    np.testing.assert_allclose(ratio.cpu().numpy(), er, rtol=1e-15 if dtype == "f64" else 1e-7)


def test_iterate_more_draws_than_the_pairwise_scan(gpu):
    """The most draws that may be compared pairwise and one more: the same values."""
    N, T = 60, 20
    h, d = columns(N, T, 1, np.float64, torch.float64)
    for B in (8192, 8193):
        seg = rng.randint(0x730, B, N)
        newlp, newval = rng.normal(0x731, T * B).astype(np.float32), rng.normal(0x732, T * B).astype(np.float32)
        value, ratio = d["value"].clone(), torch.ones(N, T, device="cuda", dtype=torch.float64)
        D.mb_iterate(D.ReplayColumns(N, T, value=value, ratio=ratio, logp=d["logp"]),
                     torch.from_numpy(seg).to("cuda", torch.int32), torch.from_numpy(newlp).cuda(),
                     torch.from_numpy(newval).cuda())
        last = {int(e): b for b, e in enumerate(seg)}
        ev = h["value"].copy()
        for e, b in last.items():
            ev[e] = newval.reshape(T, B)[:, b]
        assert np.array_equal(value.cpu().numpy(), ev)


@pytest.mark.parametrize("N,T,B", [(60, 20, 8192), (60, 256, 8192), (60, 256, 8193), (300, 255, 40), (300, 257, 40),
                                   (7, 15, 100), (3000, 16, 255), (50, 47, 4096), (50, 47, 4097), (50, 48, 4097), (50, 64, 8192),
                                   (5, 1000, 1)])
def test_iterate_forms(gpu, N, T, B):
    """Both sides of the rule between the tiles that compare draws and the last-writer table: the last draw of a
    segment leaves its values, ratios to f64's exponential, other rows untouched; invalid draws are skipped."""
    h, d = columns(N, T, 1, np.float64, torch.float64)
    seg = rng.randint(0x730 + B, B, N)
    if B > 20:
        seg[[3, 17]] = [-1, N]
    newlp, newval = rng.normal(0x731, T * B).astype(np.float32), rng.normal(0x732, T * B).astype(np.float32)
    value, ratio = d["value"].clone(), torch.ones(N, T, device="cuda", dtype=torch.float64)
    D.mb_iterate(D.ReplayColumns(N, T, value=value, ratio=ratio, logp=d["logp"]), torch.from_numpy(seg).to("cuda", torch.int32),
                 torch.from_numpy(newlp).cuda(), torch.from_numpy(newval).cuda())
    last = {int(e): b for b, e in enumerate(seg) if 0 <= e < N}
    ev, er = h["value"].copy(), np.ones((N, T))
    for e, b in last.items():
        ev[e] = newval.reshape(T, B)[:, b]
        er[e] = np.exp(newlp.reshape(T, B)[:, b].astype(np.float64) - h["logp"][e])
    assert np.array_equal(value.cpu().numpy(), ev)
    np.testing.assert_allclose(ratio.cpu().numpy(), er, rtol=1e-15)


@pytest.mark.parametrize("time_major", [True, False])
@pytest.mark.parametrize("T,B", [(1024, 1024), (1025, 1024)])
def test_gather_statistics_forms(gpu, T, B, time_major):
    """1024 blocks' partials are merged by every normalising block, more by one block: mean and std against f64. A sum of n
    terms in any tree is within a few 2^-53 sqrt(n) of exact for random signs: 1e-12."""
    N = 50
    adv = rng.normal(0x750, N * T).reshape(N, T) + 3.0
    seg = rng.randint(0x751, B, N)
    lay = lambda x: torch.from_numpy(np.ascontiguousarray(x.T if time_major else x)).cuda()
    z = lay(np.zeros((N, T)))
    cols = D.ReplayColumns(N, T, adv=lay(adv), value=z, act=z, logp=z, term=z, time_major=time_major)
    stats = torch.zeros(2, device="cuda", dtype=torch.float64)
    out = D.mb_gather(cols, torch.from_numpy(seg).to("cuda", torch.int32), stats=stats).cpu().numpy()
    a = adv[seg].T
    assert abs(stats[0].item() - a.mean()) <= 1e-12 * abs(a.mean()) and abs(stats[1].item() - a.std()) <= 1e-12 * a.std()
    np.testing.assert_allclose(out[T * B:2 * T * B].reshape(T, B), (a - a.mean()) / (a.std() + 1e-8), rtol=0, atol=1e-11)


@pytest.mark.parametrize("N,B", [(8192, 1), (8192, 129), (8193, 129), (1024, 128), (1025, 127), (1, 5), (63, 1024),
                                 (1024, 1024), (1000, 1025), (2048, 1024), (2049, 1024), (1777, 600)])
def test_sampler_edges(gpu, N, B):
    L1 = rng.randf(0x740 + N, N, 0.01, 5.0)
    seg, mp = D.prio_sample(torch.from_numpy(L1).cuda(), B, alpha=0.8, beta=0.2, rng_state=0x1234)
    idx, ref, probs, cum = O.prio_sample(L1, B, 0.8, 0.2, 0x1234)
    seg, mp = seg.cpu().numpy().astype(np.float64), mp.cpu().numpy()
    u = rng.uniform01(rng.words(0x1234, B)) * cum[-1]
    for i in np.nonzero(seg != idx)[0]:  # only a draw within rounding of a boundary, and only to its neighbour
        assert abs(seg[i] - idx[i]) == 1 and abs(cum[int(min(seg[i], idx[i]))] - u[i]) <= 1e-12 * cum[-1]
    same = seg == idx
    np.testing.assert_allclose(mp[same], ref[same], rtol=1e-12)
