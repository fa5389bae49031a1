"""The calls whose time counts: what a user of this library runs, through its public entry points.

Each case is a dict of plain values. ``listed()`` names twelve of them, ``draw(rng)`` makes more of the
same ranges, ``prepare`` builds what a program holds before the call, ``run`` is one pass, ``work`` the
bytes and operations no implementation can avoid, ``exact`` the outputs in 64 bits from plain torch and
numpy, and ``tolerance`` how far another correct implementation at the same precision may be from it.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from pufferlean_amd import _lib as L
from pufferlean_amd import device as D

GOLD = 0x9E3779B97F4A7C15
M64 = (1 << 64) - 1


def listed():
    return [
        # the trainer's MinGRU minibatch step at its full size: V-trace, forward, BPTT, clip, Muon
        dict(name="step_4096x64_h512", kind="step", B=4096, T=64, D=128, H=512, L=2, A=16, precision="bf16"),
        # the same step for a small policy in the fp32 tier, odd batch and horizon
        dict(name="step_203x33_h96_f32", kind="step", B=203, T=33, D=40, H=96, L=1, A=5, precision="f32"),
        # one environment step of the rollout: policy forward with carried state, then the sampler
        dict(name="rollout_4096_h512", kind="rollout", N=4096, D=128, H=512, L=2, A=16, precision="bf16"),
        # the smallest rollout: a few environments of a small policy (latency)
        dict(name="rollout_48_h128_f32", kind="rollout", N=48, D=24, H=128, L=1, A=6, precision="f32"),
        # the whole CartPole-sized MLP update (1024 environments x 64 steps)
        dict(name="mlp_1024x64_h128", kind="mlp", B=1024, T=64, D=4, H=128, L=2, A=2, math="bf16", muon="bf16"),
        # the host-buffer update the Lean trainer calls: two-head `target` policy, one epoch of its minibatches
        dict(name="host_update_262144", kind="host", NT=262144, D=28, H=128, heads="9,5", epochs=1, minibatches=8,
             bf16=0),
        # one dense layer, forward and both gradients (policy-sized products)
        dict(name="dense_16384x512x512", kind="dense", M=16384, K=512, N=512, dtype="bf16", math="bf16"),
        # Muon's orthogonalisation of a whole policy's matrices in one call
        dict(name="ns_6x512", kind="ns", shapes="512x512,512x512,512x512,512x512,512x1024,512x1024", math="bf16"),
        # one small odd matrix through the Muon step (tall, ragged)
        dict(name="muon_200x129", kind="muon", rows=200, cols=129, math="bf16"),
        # advantages of one rollout: V-trace on log ratios, then the normalisation
        dict(name="vtrace_4096x64", kind="vtrace", B=4096, T=64, dtype="f32", time_major=True, boot=True),
        # prioritised replay between V-trace and the BPTT on the trainer's f64 segment-major columns
        dict(name="replay_4096x64", kind="replay", N=4096, T=64, draws=4096, dtype="f64", time_major=False, K=1),
        # loss gradient of the multi-discrete head with the dashboard losses, odd row count
        dict(name="heads_md_250007", kind="heads", N=250007, mode="md", heads="9,5"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "rollout", "rollout", "mlp", "host", "dense", "dense", "ns", "muon", "vtrace",
                       "replay", "heads"])
    if kind == "step":
        H = 8 * _log(rng, 4, 64)
        c = dict(kind=kind, B=_log(rng, 16, 4096), T=_log(rng, 8, 96), D=8 * _log(rng, 1, 24), H=H,
                 L=rng.randint(1, 3), A=rng.randint(2, 17), precision=rng.choice(["bf16", "bf16", "f32"]))
        cap = 4e11 if c["precision"] == "bf16" else 4e10
        while work(c)["flops"] > cap and c["B"] > 16:
            c["B"] = max(16, c["B"] // 2)
        return c
    if kind == "rollout":
        return dict(kind=kind, N=_log(rng, 16, 8192), D=rng.randint(4, 160), H=8 * _log(rng, 8, 64), L=rng.randint(1, 3),
                    A=rng.randint(2, 24), precision=rng.choice(["bf16", "bf16", "f32"]))
    if kind == "mlp":
        m = rng.choice(["bf16", "bf16", "f32"])
        return dict(kind=kind, B=_log(rng, 32, 1024), T=_log(rng, 16, 96), D=rng.randint(3, 48),
                    H=8 * _log(rng, 4, 32), L=rng.randint(1, 3), A=rng.randint(2, 12), math=m, muon=m)
    if kind == "host":
        heads = rng.choice(["9,5", "3,3,4", "6", "5,5,2,7"])
        # few minibatches: each step orthogonalises its gradient, so a long chain amplifies a rounding
        bf, epochs = rng.choice([0, 1]), rng.randint(1, 2)
        return dict(kind=kind, NT=_log(rng, 4096, 131072), D=rng.randint(6, 48), H=8 * _log(rng, 4, 16), heads=heads,
                    epochs=epochs, minibatches=rng.choice([2, 4]) // epochs if bf else rng.choice([2, 4, 8]) // epochs,
                    bf16=bf)
    if kind == "dense":
        dt = rng.choice(["bf16", "bf16", "f32"])
        return dict(kind=kind, M=_log(rng, 256, 65536), K=_log(rng, 16, 1024), N=_log(rng, 16, 1024), dtype=dt,
                    math="bf16" if dt == "bf16" else rng.choice(["bf16", "f32"]))
    if kind == "ns":
        shapes = ["%dx%d" % (_log(rng, 16, 768), _log(rng, 16, 768)) for _ in range(rng.randint(1, 8))]
        return dict(kind=kind, shapes=",".join(shapes), math=rng.choice(["bf16", "bf16", "f32"]))
    if kind == "muon":
        return dict(kind=kind, rows=_log(rng, 4, 1536), cols=_log(rng, 16, 512), math=rng.choice(["bf16", "bf16", "f32"]))
    if kind == "vtrace":
        return dict(kind=kind, B=_log(rng, 64, 16384), T=_log(rng, 8, 256), dtype=rng.choice(["f32", "f32", "f64"]),
                    time_major=rng.choice([True, True, False]), boot=rng.choice([True, False]))
    if kind == "replay":
        dt, tm = rng.choice([("f64", False), ("f32", True)])
        return dict(kind=kind, N=_log(rng, 64, 8192), T=_log(rng, 8, 128), draws=_log(rng, 64, 4096), dtype=dt,
                    time_major=tm, K=rng.randint(1, 3))
    mode = rng.choice(["md", "cont"])
    return dict(kind="heads", N=_log(rng, 1024, 400000), mode=mode,
                heads=rng.choice(["9,5", "3,3,4", "12,7,3"]) if mode == "md" else str(rng.randint(1, 8)))


# ---- shapes ------------------------------------------------------------------------------------------
def _shapes(case):
    return [tuple(int(x) for x in s.split("x")) for s in case["shapes"].split(",")]


def _heads(case):
    return [int(x) for x in case["heads"].split(",")]


def _ns_flops(r, c, steps=5):
    m, w = min(r, c), max(r, c)
    return steps * (4.0 * m * m * w + 2.0 * m ** 3)


def _mingru_layout(c):
    """(name, rows, cols) of the flat parameters, in order; rows None for a vector."""
    H, Dm, A = c["H"], c["D"], c["A"]
    out = [("wEnc", H, Dm), ("bEnc", None, H)]
    out += [("w%d" % l, 3 * H, H) for l in range(c["L"])]
    return out + [("wDec", A, H), ("bDec", None, A), ("wVal", 1, H), ("bVal", None, 1)]


def _mlp_layout(c):
    H, O = c["H"], c["A"] + 1
    out = []
    for l in range(c["L"]):
        out += [("w%d" % l, H, c["D"] if l == 0 else H), ("b%d" % l, None, H)]
    return out + [("wo", O, H), ("bo", None, O)]


def _sizes(layout):
    return [(r or 1) * k for _, r, k in layout]


def _split(flat, layout):
    parts, off = {}, 0
    for (name, r, k), n in zip(layout, _sizes(layout)):
        v = flat[off:off + n]
        parts[name] = v.view(r, k) if r else v
        off += n
    return parts


def work(case):
    k = case["kind"]
    if k == "step":
        TB, H, Dm, A = case["T"] * case["B"], case["H"], case["D"], case["A"]
        P = sum(_sizes(_mingru_layout(case)))
        mm = TB * (H * Dm * 2.0 + case["L"] * 3.0 * H * H * 3 + (A + 1) * H * 3.0)
        ns = sum(_ns_flops(r, c) for _, r, c in _mingru_layout(case) if r)
        return {"bytes": 4.0 * TB * (Dm + 6) + 4.0 * 5 * P, "flops": 2.0 * mm + ns}
    if k == "rollout":
        N, H, Dm, A, Ln = case["N"], case["H"], case["D"], case["A"], case["L"]
        P = H * Dm + H + Ln * 3 * H * H + (A + 1) * (H + 1)
        return {"bytes": 4.0 * (P + N * Dm + 2 * N * Ln * H + N * (A + 4)),
                "flops": 2.0 * N * (H * Dm + Ln * 3 * H * H + (A + 1) * H)}
    if k == "mlp":
        N = case["B"] * case["T"]
        mats = [(r, c) for _, r, c in _mlp_layout(case) if r]
        P = sum(_sizes(_mlp_layout(case)))
        fl = sum(r * c for r, c in mats) * 6.0 * N - 2.0 * N * mats[0][0] * mats[0][1]
        return {"bytes": 4.0 * N * (case["D"] + 4) + 4.0 * 5 * P, "flops": fl + sum(_ns_flops(r, c) for r, c in mats)}
    if k == "host":
        hs, NT, H, Dm, E = _heads(case), case["NT"], case["H"], case["D"], case["epochs"]
        O = sum(hs) + 1
        per = 2.0 * (2 * H * Dm + 3 * H * O)
        return {"bytes": 8.0 * NT * (Dm + len(hs) + 4 + E) + 32.0 * (H * Dm + H + O * H + O),
                "flops": per * NT * E + E * case["minibatches"] * (_ns_flops(H, Dm) + _ns_flops(O, H))}
    if k == "dense":
        M, K, N = case["M"], case["K"], case["N"]
        e = 2.0 if case["dtype"] == "bf16" else 4.0
        return {"bytes": e * (2 * M * K + 2 * M * N + N * K) + 4.0 * (N * K + N), "flops": 6.0 * M * N * K}
    if k == "ns":
        return {"bytes": sum(8.0 * r * c for r, c in _shapes(case)), "flops": sum(_ns_flops(r, c) for r, c in _shapes(case))}
    if k == "muon":
        r, c = case["rows"], case["cols"]
        return {"bytes": 20.0 * r * c, "flops": _ns_flops(r, c) + 8.0 * r * c}
    if k == "vtrace":
        n, e = case["B"] * case["T"], 8.0 if case["dtype"] == "f64" else 4.0
        return {"bytes": e * (7 * n + (case["B"] if case["boot"] else 0)), "flops": 18.0 * n}
    if k == "replay":
        e, n, nd = 8.0 if case["dtype"] == "f64" else 4.0, case["N"] * case["T"], case["draws"] * case["T"]
        K = case["K"]
        return {"bytes": e * n + nd * e * (4 + K) + nd * e * (5 + K) + nd * 8.0 + 3 * e * min(n, nd) + 28.0 * case["draws"],
                "flops": 12.0 * nd}
    N, hs = case["N"], _heads(case)
    O, Wd = (sum(hs) + 1, len(hs)) if case["mode"] == "md" else (2 * hs[0] + 1, hs[0])
    return {"bytes": 4.0 * N * (2 * O + Wd + 6), "flops": 20.0 * N * O}


# Relative 2-norm errors: about four times the largest seen against exact() over the listed cases and 600
# drawn ones (largest seen in the comment). 16-bit products: a rounding moves rows whose ratio lies on a clip edge
# to the other branch, which dominates the step's and, over a chain of minibatches, the host update's figure.
_TOL = {
    ("step", "bf16"): 1e-1,     # 4.7e-2 (gradient of a small policy with clip flips; 1.7e-3 without)
    ("step", "f32"): 7e-5,      # 1.7e-5
    ("rollout", "bf16"): 2e-2,  # 4.8e-3 (outputs); draws below
    ("rollout", "f32"): 2e-6,   # 5.4e-7
    ("mlp", "bf16"): 6e-3,      # 1.4e-3
    ("mlp", "f32"): 2.5e-5,     # 6.0e-6
    ("host", 1): 1.6e-1,        # 4.2e-2 (momentum after four minibatches)
    ("host", 0): 4e-2,          # 1.1e-2 (one row's clip edge, amplified over eight; 1e-6 to 5e-4 without)
    ("dense", "bf16"): 1e-2,    # 2.4e-3
    ("dense", "f32"): 2e-6,     # 5.4e-7
    ("ns", "bf16"): 2e-2,       # 7.3e-3
    ("ns", "f32"): 1e-5,        # 2.6e-6
    ("muon", "bf16"): 4e-4,     # 9.4e-5 of the weight, whose step is a few per cent of it
    ("muon", "f32"): 2e-7,      # 3.2e-8
    ("vtrace", "f32"): 8e-7,    # 2.0e-7
    ("vtrace", "f64"): 1e-15,   # 2.4e-16
    ("replay", "f32"): 2e-7,    # 2.6e-8
    ("replay", "f64"): 1e-14,   # 8.8e-17
    ("heads", "f32"): 6e-6,     # 1.4e-6
}


def tolerance(case):
    k = case["kind"]
    tier = {"step": "precision", "rollout": "precision", "mlp": "math", "host": "bf16", "dense": "math", "ns": "math",
            "muon": "math", "vtrace": "dtype", "replay": "dtype"}.get(k)
    t = {"rel": _TOL[(k, case[tier] if tier else "f32")]}
    if k == "rollout":
        # a draw within rounding of a cumulative boundary takes the neighbouring action (0.4 % of bf16 rows seen,
        # never in fp32), and its log-prob is that action's: two such rows, or 1 %, are within tolerance
        bf = case["precision"] == "bf16"
        t["differ"] = max(1e-2 if bf else 1e-4, 2.0 / case["N"])
        if bf:
            t["rel"] = max(t["rel"], 0.5 * math.sqrt(t["differ"]))
    if k == "replay":
        t["differ"] = max(1e-4, 1.0 / case["draws"])
    return t


# ---- inputs ------------------------------------------------------------------------------------------
class _Gen:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFFFFFFFFFF)

    def normal(self, *shape, std=1.0, mean=0.0):
        return torch.randn(*shape, generator=self.g, device="cuda") * std + mean

    def uniform(self, *shape):
        return torch.rand(*shape, generator=self.g, device="cuda")

    def ints(self, hi, *shape):
        return torch.randint(0, hi, shape, generator=self.g, device="cuda", dtype=torch.int32)

    def flags(self, p, *shape):
        return (self.uniform(*shape) < p).float()


def _flat_params(g, layout, heads=()):
    """N(0, 1/fan_in) weights, zero biases; a policy head starts near uniform (a tenth of that)."""
    parts = []
    for name, r, k in layout:
        if r:
            parts.append((g.normal(r * k) * ((0.1 if name in heads else 1.0) / math.sqrt(k))))
        else:
            parts.append(torch.zeros(k, device="cuda"))
    return torch.cat(parts)


class _Policy:
    """A resident policy handle ([params; momentum] in f64 on the device), freed with the state."""

    def __init__(self, pm):
        self.P = pm.size // 2
        self.h = C.c_size_t(0)
        L.call("ph_cuda_policy_load", _dp(pm), self.P, C.byref(self.h))

    def __del__(self):
        L.call("ph_cuda_policy_free", self.h.value)


def _dp(a):
    return a.ctypes.data_as(L.dptr)


def _inputs(case, seed):
    """The tensors (numpy arrays for the host entry) of the call, from the seed alone."""
    k, g, s = case["kind"], None, {}
    if k != "host":
        g = _Gen(seed)
    if k == "step":
        T, B, A = case["T"], case["B"], case["A"]
        s["params"] = _flat_params(g, _mingru_layout(case), heads=("wDec",))
        s["mom"] = torch.zeros_like(s["params"])
        s["obs"] = g.normal(T, B, case["D"])
        s["act"] = g.ints(A, T, B)
        s["old"] = g.normal(T, B, std=0.05, mean=math.log(1.0 / A))
        s["val"], s["rew"] = g.normal(T, B), g.normal(T, B)
        s["done"], s["logrho"] = g.flags(0.01, T, B), g.normal(T, B, std=0.1)
        s["boot"] = g.normal(B)
    elif k == "rollout":
        N = case["N"]
        s["params"] = _flat_params(g, _mingru_layout(case))
        s["obs"] = g.normal(N, case["D"])
        s["state"] = g.normal(N, case["L"], case["H"], std=0.5)
        s["rng"] = int(seed) * 0x2545F4914F6CDD1D & M64
    elif k == "mlp":
        N, A = case["B"] * case["T"], case["A"]
        s["params"] = _flat_params(g, _mlp_layout(case), heads=("wo",))
        s["mom"] = torch.zeros_like(s["params"])
        s["obs"] = g.uniform(N, case["D"]) * 2 - 1
        s["act"] = g.ints(A, N)
        s["old"] = g.normal(N, std=0.05, mean=math.log(1.0 / A))
        s["rew"], s["done"] = g.normal(N, std=0.5, mean=0.5), g.flags(0.02, N)
    elif k == "host":
        r = np.random.default_rng(int(seed) & M64)
        hs, NT, H, Dm = _heads(case), case["NT"], case["H"], case["D"]
        O = sum(hs) + 1
        w1, w2 = r.standard_normal(H * Dm) / math.sqrt(Dm), r.standard_normal(O * H) * (0.1 / math.sqrt(H))
        par = np.concatenate([w1, np.zeros(H), w2, np.zeros(O)])
        s["pm"] = np.concatenate([par, np.zeros_like(par)])
        s["obs"] = r.standard_normal(NT * Dm)
        s["acts"] = np.stack([r.integers(0, h, NT) for h in hs], 1).astype(np.float64).ravel()
        s["adv"], s["ret"], s["ov"] = r.standard_normal(NT), r.standard_normal(NT) * 0.5, r.standard_normal(NT) * 0.2
        s["olp"] = -math.log(math.prod(hs)) + 0.05 * r.standard_normal(NT)
        s["perm"] = np.concatenate([r.permutation(NT) for _ in range(case["epochs"])]).astype(np.float64)
        s["hs"] = np.array(hs, np.float64)
    elif k == "dense":
        M, K, N = case["M"], case["K"], case["N"]
        dt = torch.bfloat16 if case["dtype"] == "bf16" else torch.float32
        s["x"], s["w"] = g.normal(M, K).to(dt), (g.normal(N, K) / math.sqrt(K)).to(dt)
        s["b"], s["dy"] = g.normal(N, std=0.1), g.normal(M, N).to(dt)
    elif k == "ns":
        s["mats"] = [g.normal(r, c, std=0.02) for r, c in _shapes(case)]
    elif k == "muon":
        r, c = case["rows"], case["cols"]
        s["w"], s["grad"], s["mom"] = g.normal(r, c, std=1 / math.sqrt(c)), g.normal(r, c, std=0.01), g.normal(r, c, std=0.05)
    elif k == "vtrace":
        shape = (case["T"], case["B"]) if case["time_major"] else (case["B"], case["T"])
        dt = torch.float64 if case["dtype"] == "f64" else torch.float32
        s["rew"], s["val"] = g.normal(*shape).to(dt), g.normal(*shape).to(dt)
        s["done"], s["logrho"] = g.flags(0.01, *shape).to(dt), g.normal(*shape, std=0.1).to(dt)
        s["boot"] = g.normal(case["B"]).to(dt) if case["boot"] else None
    elif k == "replay":
        N, T, K = case["N"], case["T"], case["K"]
        dt = torch.float64 if case["dtype"] == "f64" else torch.float32
        shape = (T, N) if case["time_major"] else (N, T)
        s["adv"], s["value"] = g.normal(*shape).to(dt), g.normal(*shape).to(dt)
        s["logp"], s["term"] = g.normal(*shape, std=0.3, mean=-2.0).to(dt), g.flags(0.01, *shape).to(dt)
        s["act"] = g.ints(8, *shape, K).to(dt)
        s["newlp"], s["newval"] = g.normal(T, case["draws"], std=0.3, mean=-2.0), g.normal(T, case["draws"])
        s["rng"] = int(seed) * 0x2545F4914F6CDD1D & M64
    else:
        N, hs = case["N"], _heads(case)
        if case["mode"] == "md":
            s["out"] = g.normal(N, sum(hs) + 1)
            s["act"] = torch.stack([g.ints(h, N) for h in hs], 1).contiguous()
            s["old"] = g.normal(N, std=0.3, mean=-math.log(math.prod(hs)))
        else:
            d = hs[0]
            s["out"] = torch.cat([g.normal(N, d), g.normal(N, d, std=0.3, mean=-0.5), g.normal(N, 1)], 1).contiguous()
            s["act"] = (s["out"][:, :d] + g.normal(N, d) * s["out"][:, d:2 * d].exp()).contiguous()
            s["old"] = g.normal(N, std=0.5, mean=-0.9 * d)
        s["adv"], s["ret"], s["ov"] = g.normal(N), g.normal(N), g.normal(N)
    return s


def prepare(case, seed):
    k, s = case["kind"], _inputs(case, seed)
    s["case"] = case
    if k == "step":
        s["cfg"] = D.MinGRUConfig(case["B"], case["T"], case["D"], case["H"], case["L"], case["A"], lr=0.015, mu=0.95,
                                  max_grad_norm=0.5, gscale=1.0 / (case["B"] * case["T"]), precision=case["precision"],
                                  math=case["precision"])
        s["G"] = torch.zeros_like(s["params"])
    elif k == "rollout":
        N = case["N"]
        s["out"] = torch.empty(N, case["A"] + 1, device="cuda")
        s["act"] = torch.empty(N, device="cuda", dtype=torch.int32)
        s["logp"], s["value"] = torch.empty(N, device="cuda"), torch.empty(N, device="cuda")
    elif k == "mlp":
        s["cfg"] = D.MLPConfig(case["B"] * case["T"], case["D"], case["H"], case["L"], case["A"], lr=0.015,
                               max_grad_norm=0.5, math=case["math"], muon_math=case["muon"])
        s["G"] = torch.empty_like(s["params"])
    elif k == "host":
        s["policy"] = _Policy(s.pop("pm"))
        s["peek"], s["back"] = np.zeros(1), np.zeros(2 * s["policy"].P)
    elif k == "dense":
        dt = s["x"].dtype
        s["y"] = torch.empty(case["M"], case["N"], device="cuda", dtype=dt)
        s["dx"] = torch.empty(case["M"], case["K"], device="cuda", dtype=dt)
        s["dw"] = torch.empty(case["N"], case["K"], device="cuda")
    elif k == "ns":
        s["work"] = [torch.empty_like(m) for m in s["mats"]]
    elif k == "vtrace":
        s["advn"], s["tgt"], s["raw"] = (torch.empty_like(s["rew"]) for _ in range(3))
    elif k == "replay":
        s["ratio"] = torch.ones_like(s["value"])
        s["cols"] = D.ReplayColumns(case["N"], case["T"], adv=s["adv"], value=s["value"], ratio=s["ratio"], act=s["act"],
                                    logp=s["logp"], term=s["term"], time_major=case["time_major"], K=case["K"])
        Bd = case["draws"]
        s["L1"] = torch.empty(case["N"], device="cuda", dtype=torch.float64)
        s["seg"] = torch.empty(Bd, device="cuda", dtype=torch.int32)
        s["mp"] = torch.empty(Bd, device="cuda", dtype=torch.float64)
        s["mb"] = torch.empty((case["K"] + 5) * case["T"] * Bd, device="cuda", dtype=s["value"].dtype)
    elif k == "heads":
        s["dout"] = torch.empty_like(s["out"])
        s["newlp"], s["newval"] = torch.empty(case["N"], device="cuda"), torch.empty(case["N"], device="cuda")
        s["losses"] = torch.zeros(7, device="cuda", dtype=torch.float64)
    return s


def run(s):
    case = s["case"]
    k = case["kind"]
    if k == "step":
        D.mingru_step(s["cfg"], s["params"], s["mom"], s["obs"], s["act"], s["old"], s["val"], s["rew"], s["done"],
                      s["logrho"], s["boot"], G=s["G"])
        return {"params": s["params"], "mom": s["mom"], "G": s["G"]}
    if k == "rollout":
        D.mingru_rollout_step(s["params"], s["obs"], s["state"], s["out"], D=case["D"], H=case["H"], L_layers=case["L"],
                              A=case["A"], precision=0 if case["precision"] == "bf16" else 1)
        D.sample_actions(s["out"], case["A"], rng_state=s["rng"], act=s["act"], logp=s["logp"], value=s["value"])
        s["rng"] = (s["rng"] + case["N"] * GOLD) & M64
        return {"out": s["out"], "state": s["state"], "act": s["act"], "logp": s["logp"], "value": s["value"]}
    if k == "mlp":
        D.mlp_update(s["cfg"], case["T"], s["params"], s["mom"], s["obs"], s["act"], s["old"], s["rew"], s["done"], G=s["G"])
        return {"params": s["params"], "mom": s["mom"], "G": s["G"]}
    if k == "host":
        hs, p = _heads(case), s["policy"]
        L.call("ph_cuda_train_update_wide_resident", p.h.value, _dp(s["obs"]), _dp(s["acts"]), _dp(s["adv"]), _dp(s["ret"]),
               _dp(s["olp"]), _dp(s["ov"]), case["NT"], _dp(s["perm"]), _dp(s["hs"]), len(hs), case["NT"], case["D"],
               case["H"], sum(hs) + 1, len(hs), 1, case["epochs"], case["minibatches"], 0.015, 0.0, 0.95, 1e-12, 2.0,
               0.001, 0.2, 0.2, 1.5, case["bf16"], _dp(s["peek"]))
        L.call("ph_cuda_policy_download", p.h.value, p.P, _dp(s["back"]))
        return {"params": s["back"][:p.P], "mom": s["back"][p.P:]}
    if k == "dense":
        D.gemm(s["x"], s["w"], trans_b=True, out=s["y"], math=case["math"], epilogue=L.PH_EPI_BIAS_RELU, bias=s["b"])
        D.gemm(s["dy"], s["w"], out=s["dx"], math=case["math"])
        D.gemm(s["dy"], s["x"], trans_a=True, out=s["dw"], math=case["math"])
        return {"y": s["y"], "dx": s["dx"], "dw": s["dw"]}
    if k == "ns":
        for w, m in zip(s["work"], s["mats"]):
            w.copy_(m)  # the entry works in place; a program orthogonalises its momentum's copy
        D.newton_schulz_batch(s["work"], math=case["math"])
        return list(s["work"])
    if k == "muon":
        D.muon_mat(s["w"], s["grad"], s["mom"], math=case["math"])
        return {"w": s["w"], "mom": s["mom"]}
    if k == "vtrace":
        D.vtrace(s["rew"], s["val"], s["done"], s["logrho"], s["boot"], variant=1 if case["boot"] else 0,
                 time_major=case["time_major"], rho_is_log=True, out_adv=s["raw"], out_tgt=s["tgt"])
        D.adv_normalize(s["raw"], out=s["advn"])
        return {"adv": s["raw"], "tgt": s["tgt"], "advn": s["advn"]}
    if k == "replay":
        D.seg_l1(s["cols"], out=s["L1"])
        D.prio_sample(s["L1"], case["draws"], alpha=0.8, beta=0.2, rng_state=s["rng"], seg=s["seg"], mbprio=s["mp"])
        D.mb_gather(s["cols"], s["seg"], s["mp"], out=s["mb"])
        D.mb_iterate(s["cols"], s["seg"], s["newlp"], s["newval"])
        s["rng"] = (s["rng"] + case["draws"] * GOLD) & M64
        return {"L1": s["L1"], "seg": s["seg"], "mbprio": s["mp"], "mb": s["mb"], "value": s["value"], "ratio": s["ratio"]}
    kw = dict(vf_clip=0.2, dout=s["dout"], newlp=s["newlp"], newval=s["newval"], losses=s["losses"])
    if case["mode"] == "md":
        D.ppo_grad_md(s["out"], s["act"], s["adv"], s["ret"], s["old"], s["ov"], head_sizes=_heads(case), **kw)
    else:
        D.ppo_grad_cont(s["out"], s["act"], s["adv"], s["ret"], s["old"], s["ov"], dim=_heads(case)[0], **kw)
    return {"dout": s["dout"], "newlp": s["newlp"], "newval": s["newval"], "losses": s["losses"]}


# ---- the same in 64 bits -----------------------------------------------------------------------------
def _f32(x):
    return float(np.float32(x))


def _ns64(X, coeffs, eps=_f32(1e-7)):
    t = X.shape[0] > X.shape[1]
    Y = X.t() if t else X
    Y = Y / (Y.norm() + eps)
    for a, b, c in coeffs:
        G = Y @ Y.t()
        Y = a * Y + (b * G + c * (G @ G)) @ Y
    return Y.t() if t else Y


CONST64 = [tuple(_f32(x) for x in row) for row in D.CONST_COEFFS]


def _muon64(w, g, m, lr, mu, coeffs, eps):
    """One Muon step of a matrix (or, for a vector, Nesterov momentum): (w, m)."""
    m = mu * m + g
    u = g + mu * m
    if w.dim() == 1:
        return w + lr * u, m
    return w + lr * math.sqrt(max(1.0, w.shape[0] / w.shape[1])) * _ns64(u, coeffs, eps), m


def _opt64(params, mom, G, layout, lr, mu, coeffs, eps):
    w, g, m = (_split(x, layout) for x in (params, G, mom))
    new = [_muon64(w[n], g[n], m[n], lr, mu, coeffs, eps) for n, _, _ in layout]
    return torch.cat([a.reshape(-1) for a, _ in new]), torch.cat([b.reshape(-1) for _, b in new])


def _clip64(G, scale, max_norm):
    G = G * scale
    n = float(G.norm())
    return G * (max_norm / n if max_norm > 0 and n > max_norm else 1.0)


def _vtrace64(rew, val, done, logrho, boot, gamma, lam):
    """Time-major reverse scan with unit clips: (advantages, targets)."""
    T, B = rew.shape
    adv = torch.zeros_like(rew)
    last = torch.zeros_like(rew[0])
    for t in range(T - 1, -1, -1):
        if boot is None and t == T - 1:
            continue
        w = logrho[t].exp().clamp(max=1.0)
        nv = boot if t == T - 1 else val[t + 1]
        nnt = 1.0 - (done[t] > 0.5).to(rew.dtype)
        r = rew[t].clamp(-1, 1)
        d = w * (r + gamma * nv * nnt - val[t]) if boot is None else w * r + gamma * nv * nnt - val[t]
        last = d + gamma * lam * w * last * nnt
        adv[t] = last
    return adv, adv + val


def _norm64(a):
    return (a - a.mean()) / (a.std(unbiased=False) + 1e-8)


def _vloss64(v, ret, ov, vclip):
    du = (v - ret) ** 2
    if ov is None or vclip <= 0:
        return 0.5 * du
    vc = ov + (v - ov).clamp(-vclip, vclip)
    return 0.5 * torch.maximum(du, (vc - ret) ** 2)


def _ppo64(logp, ent, v, adv, ret, old, ov=None, vf=_f32(0.5), entc=_f32(0.01), clip=_f32(0.2), vclip=0.0):
    """The summed PPO objective (its gradient is the ascent gradient)."""
    r = (logp - old).exp()
    pg = torch.minimum(adv * r, adv * r.clamp(1 - clip, 1 + clip))
    return (pg + entc * ent - vf * _vloss64(v, ret, ov, vclip)).sum()


def _cat64(logits, act):
    ls = logits.log_softmax(-1)
    return ls.gather(-1, act.long().unsqueeze(-1)).squeeze(-1), -(ls.exp() * ls).sum(-1)


def _gact(x):
    return torch.where(x >= 0, x + 0.5, torch.sigmoid(x))


def _exact_step(case, s):
    f = lambda x: x.double()
    lay = _mingru_layout(case)
    T, B, H = case["T"], case["B"], case["H"]
    adv, tgt = _vtrace64(f(s["rew"]), f(s["val"]), f(s["done"]), f(s["logrho"]), f(s["boot"]), _f32(0.99), _f32(0.95))
    p = f(s["params"]).requires_grad_(True)
    w = _split(p, lay)
    x = f(s["obs"]).view(T * B, -1) @ w["wEnc"].t() + w["bEnc"]
    keep = (s["done"] == 0).double().unsqueeze(-1)
    for l in range(case["L"]):
        hid, gate, proj = (x @ w["w%d" % l].t()).view(T, B, 3, H).unbind(2)
        z, cand, hg = torch.sigmoid(gate), _gact(hid), torch.sigmoid(proj)
        st, os = torch.zeros(B, H, device="cuda", dtype=torch.float64), []
        for t in range(T):
            o = (1 - z[t]) * st + z[t] * cand[t]
            os.append(o)
            st = o * keep[t]
        x = (hg * torch.stack(os) + (1 - hg) * x.view(T, B, H)).view(T * B, H)
    v = (x @ w["wVal"].t() + w["bVal"]).view(-1)
    lp, ent = _cat64(x @ w["wDec"].t() + w["bDec"], s["act"].view(-1))
    obj = _ppo64(lp, ent, v, _norm64(adv).view(-1), tgt.view(-1), f(s["old"]).view(-1))
    (G,) = torch.autograd.grad(obj, p)
    G = _clip64(G, _f32(1.0 / (T * B)), 0.5)
    par, mom = _opt64(p.detach(), f(s["mom"]), G, lay, _f32(0.015), _f32(0.95), CONST64, _f32(1e-7))
    return {"params": par, "mom": mom, "G": G}


def _exact_mlp(case, s):
    f = lambda x: x.double()
    lay, T, B = _mlp_layout(case), case["T"], case["B"]
    p = f(s["params"]).requires_grad_(True)
    w = _split(p, lay)
    x = f(s["obs"])
    for l in range(case["L"]):
        x = torch.relu(x @ w["w%d" % l].t() + w["b%d" % l])
    out = x @ w["wo"].t() + w["bo"]
    lp, ent = _cat64(out[:, :case["A"]], s["act"])
    v, old = out[:, case["A"]], f(s["old"])
    tm = lambda x: x.detach().view(T, B)
    adv, tgt = _vtrace64(tm(f(s["rew"])), tm(v), tm(f(s["done"])), tm(lp - old), None, _f32(0.99), _f32(0.95))
    obj = _ppo64(lp, ent, v, _norm64(adv).view(-1), tgt.view(-1), old)
    (G,) = torch.autograd.grad(obj, p)
    G = _clip64(G, _f32(1.0 / (T * B)), 0.5)
    par, mom = _opt64(p.detach(), f(s["mom"]), G, lay, _f32(0.015), _f32(0.95), CONST64, _f32(1e-7))
    return {"params": par, "mom": mom, "G": G}


def _exact_host(case, s):
    hs, NT, Dm, H = _heads(case), case["NT"], case["D"], case["H"]
    O, nmb = sum(hs) + 1, case["minibatches"]
    c = lambda x: torch.from_numpy(x).cuda()
    lay = [("w1", H, Dm), ("b1", None, H), ("w2", O, H), ("b2", None, O)]
    obs, acts = c(s["obs"]).view(NT, Dm), c(s["acts"]).view(NT, -1)
    adv, ret, old, ov = (c(s[n]) for n in ("adv", "ret", "olp", "ov"))
    pm = c(s["pm"])
    par, mom = pm[:pm.numel() // 2].clone(), pm[pm.numel() // 2:].clone()
    perm = c(s["perm"]).long().view(case["epochs"], NT)
    mb = NT // nmb
    for e in range(case["epochs"]):
        for m in range(nmb):
            ix = perm[e, m * mb:(NT if m + 1 == nmb else (m + 1) * mb)]
            p = par.clone().requires_grad_(True)
            w = _split(p, lay)
            out = torch.relu(obs[ix] @ w["w1"].t() + w["b1"]) @ w["w2"].t() + w["b2"]
            parts = [_cat64(l, acts[ix, h]) for h, l in enumerate(out[:, :O - 1].split(hs, dim=1))]
            obj = _ppo64(sum(a for a, _ in parts), sum(b for _, b in parts), out[:, O - 1], _norm64(adv[ix]), ret[ix],
                         old[ix], ov[ix], 2.0, 0.001, 0.2, 0.2)
            (G,) = torch.autograd.grad(obj, p)
            par, mom = _opt64(par, mom, _clip64(G, 1.0 / len(ix), 1.5), lay, 0.015, 0.95, D.REF_COEFFS, 1e-12)
    return {"params": par.cpu().numpy(), "mom": mom.cpu().numpy()}


def _words(state):
    with np.errstate(over="ignore"):
        z = state
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        return z ^ (z >> np.uint64(31))


def _uniforms(rng, n):
    with np.errstate(over="ignore"):
        w = _words(np.uint64(rng) + np.arange(1, n + 1, dtype=np.uint64) * np.uint64(GOLD))
    return (w >> np.uint64(11)).astype(np.float64) / 9007199254740992.0


def _exact_rollout(case, s):
    f = lambda x: x.double()
    w = _split(f(s["params"]), _mingru_layout(case))
    x, st = f(s["obs"]) @ w["wEnc"].t() + w["bEnc"], f(s["state"])
    new = []
    for l in range(case["L"]):
        hid, gate, proj = (x @ w["w%d" % l].t()).chunk(3, 1)
        z, hg = torch.sigmoid(gate), torch.sigmoid(proj)
        o = (1 - z) * st[:, l] + z * _gact(hid)
        new.append(o)
        x = hg * o + (1 - hg) * x
    out = torch.cat([x @ w["wDec"].t() + w["bDec"], x @ w["wVal"].t() + w["bVal"]], 1)
    ls = out[:, :-1].log_softmax(1)
    u = torch.from_numpy(_uniforms(s["rng"], case["N"])).cuda()
    act = (ls.exp().cumsum(1) <= u.unsqueeze(1)).sum(1).clamp(max=case["A"] - 1)
    return {"out": out, "state": torch.stack(new, 1), "act": act.int(), "logp": ls.gather(1, act.unsqueeze(1)).squeeze(1),
            "value": out[:, -1]}


def _exact_replay(case, s):
    N, T, Bd, K = case["N"], case["T"], case["draws"], case["K"]
    col = lambda x: (x.double().transpose(0, 1) if case["time_major"] else x.double())  # [N, T]
    adv, val, logp, term, act = (col(s[n]) for n in ("adv", "value", "logp", "term", "act"))
    L1 = adv.abs().sum(1)
    p = (0.8 * (L1 + 1e-12).log()).exp()
    p = (p + 1e-6) / (p.sum() + 1e-6)
    cum = p.cumsum(0)
    u = torch.from_numpy(_uniforms(s["rng"], Bd)).cuda() * p.sum()
    seg = torch.searchsorted(cum, u).clamp(max=N - 1)
    mp = (-0.2 * (N * p[seg] + 1e-12).log()).exp()
    a = adv[seg]
    an = mp.unsqueeze(1) * ((a - a.mean()) / (a.std(unbiased=False) + 1e-8))
    tm = lambda x: x.transpose(0, 1).reshape(-1)  # [Bd, T] -> timestep-major
    mb = torch.cat([act[seg].transpose(0, 1).reshape(-1), tm(an), tm(a + val[seg]), tm(logp[seg]),
                    tm((term[seg] > 0.5).double()), tm(val[seg])])
    last = torch.full((N,), -1, device="cuda", dtype=torch.int64)
    last.scatter_reduce_(0, seg, torch.arange(Bd, device="cuda"), "amax")
    hit = last >= 0
    value, ratio = val.clone(), torch.ones_like(val)
    value[hit] = s["newval"].double()[:, last[hit]].t()
    ratio[hit] = (s["newlp"].double()[:, last[hit]].t() - logp[hit]).exp()
    back = lambda x: (x.transpose(0, 1).contiguous() if case["time_major"] else x)
    return {"L1": L1, "seg": seg.int(), "mbprio": mp, "mb": mb, "value": back(value), "ratio": back(ratio)}


def _exact_heads(case, s):
    f = lambda x: x.double()
    hs, adv, ret, old, ov = _heads(case), f(s["adv"]), f(s["ret"]), f(s["old"]), f(s["ov"])
    o = f(s["out"]).requires_grad_(True)
    if case["mode"] == "md":
        parts = [_cat64(l, s["act"][:, h]) for h, l in enumerate(o[:, :-1].split(hs, dim=1))]
        lp, ent = sum(a for a, _ in parts), sum(b for _, b in parts)
        c = 0.0
    else:
        d = hs[0]
        c = 0.5 * math.log(2 * math.pi)
        raw = o[:, d:2 * d]
        ls = raw.clamp(-20.0, 2.0)
        z = (f(s["act"]) - o[:, :d]) * (-ls).exp()
        lp, ent = (-0.5 * z * z - ls - c).sum(1), (ls + 0.5 + c).sum(1)
    v, clip = o[:, -1], _f32(0.2)
    (dout,) = torch.autograd.grad(_ppo64(lp, ent, v, adv, ret, old, ov, vclip=_f32(0.2)), o)
    with torch.no_grad():
        lr = lp - old
        r = lr.exp()
        pg = torch.maximum(-adv * r, -adv * r.clamp(1 - clip, 1 + clip)).mean()
        vl, en = _vloss64(v, ret, ov, _f32(0.2)).mean(), ent.mean()
        cf = ((r < 1 - clip) | (r > 1 + clip)).double().mean()
        losses = torch.stack([pg, vl, en, pg + _f32(0.5) * vl - _f32(0.01) * en, -lr.mean(), (r - 1 - lr).mean(), cf])
    return {"dout": dout, "newlp": lp.detach(), "newval": v.detach(), "losses": losses}


def exact(case, seed):
    k, s = case["kind"], _inputs(case, seed)
    f = lambda x: x.double()
    if k == "step":
        return _exact_step(case, s)
    if k == "rollout":
        return _exact_rollout(case, s)
    if k == "mlp":
        return _exact_mlp(case, s)
    if k == "host":
        return _exact_host(case, s)
    if k == "dense":
        x, w, dy = f(s["x"]), f(s["w"]), f(s["dy"])
        return {"y": torch.relu(x @ w.t() + f(s["b"])), "dx": dy @ w, "dw": dy.t() @ x}
    if k == "ns":
        return [_ns64(f(m), CONST64) for m in s["mats"]]
    if k == "muon":
        w, m = _muon64(f(s["w"]), f(s["grad"]), f(s["mom"]), _f32(0.015), _f32(0.95), CONST64, _f32(1e-7))
        return {"w": w, "mom": m}
    if k == "vtrace":
        tm = (lambda x: f(x)) if case["time_major"] else (lambda x: f(x).t())
        adv, tgt = _vtrace64(tm(s["rew"]), tm(s["val"]), tm(s["done"]), tm(s["logrho"]),
                             f(s["boot"]) if case["boot"] else None, 0.99, 0.95)
        back = (lambda x: x) if case["time_major"] else (lambda x: x.t().contiguous())
        return {"adv": back(adv), "tgt": back(tgt), "advn": back(_norm64(adv))}
    if k == "replay":
        return _exact_replay(case, s)
    return _exact_heads(case, s)
