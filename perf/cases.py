"""Timed workloads of flowmc_amd: the calls that a sampling run is made of.

A run alternates local steps (fused MALA / HMC / random-walk chains, batched
HMC over several targets, parallel tempering), global steps (proposals from a
normalizing flow and their Metropolis-Hastings scan) and flow training. Every
case is one such call through the strategy, kernel or model that a program
calls, from the smallest runs (20 chains, a few dimensions, default flow) to
the 64-dimensional mixture with 4096 chains and its 409,600 proposals a step.

``exact`` computes the same results in FP64 with plain torch: the random
numbers are the Philox4x32-10 streams that the keys stand for, redrawn here.
"""

import math

import numpy as np
import torch

from flowmc_amd import random as fr
from flowmc_amd import targets as TG
from flowmc_amd.resource.buffers import Buffer
from flowmc_amd.resource.kernel.batched_HMC import BatchedHMC
from flowmc_amd.resource.kernel.Gaussian_random_walk import GaussianRandomWalk
from flowmc_amd.resource.kernel.HMC import HMC
from flowmc_amd.resource.kernel.MALA import MALA
from flowmc_amd.resource.kernel.NF_proposal import NFProposal
from flowmc_amd.resource.logPDF import LogPDF, TemperedPDF
from flowmc_amd.resource.model.nf_model.realNVP import RealNVP
from flowmc_amd.resource.model.nf_model.rqSpline import MaskedCouplingRQSpline
from flowmc_amd.resource.optimizer import AdamState, AdamWClip
from flowmc_amd.resource.states import State
from flowmc_amd.strategy.parallel_tempering import ParallelTempering
from flowmc_amd.strategy.take_steps import TakeGroupSteps, TakeSerialSteps

DEV = "cuda"
F64 = torch.float64


# ------------------------------------------------------------------ cases --
def listed():
    return [
        # Local steps of the usual small run: a correlated 5-D Gaussian, 1000
        # chains, one long call. A step's serial chain is what it waits for.
        dict(name="mala_gauss5d", kind="local", kernel="mala", target="gauss", dim=5, chains=1000, steps=1000,
             thinning=1, step_size=0.1),
        # The throughput end of local sampling: 16384 chains, every row kept.
        dict(name="mala_rosenbrock128d", kind="local", kernel="mala", target="rosenbrock", dim=128, chains=16384,
             steps=64, thinning=1, step_size=0.01),
        # 32 funnels of uneven dimension advanced by one launch.
        dict(name="hmc_funnels", kind="batched_hmc", targets=32, lo=8, hi=256, chains=256, steps=16, leapfrog=10,
             step_size=0.05),
        # One parallel-tempering call in training: tempered MALA on the 8-mode
        # 64-D mixture, swap sweep, ladder adaptation.
        dict(name="tempering_gmm64d", kind="tempering", dim=64, modes=8, chains=4096, temps=5, steps=100,
             step_size=0.05),
        # The global step of the quickstart's size: 20 chains, 50 proposals
        # each, the default flow. Launches and latency are all of it.
        dict(name="global_step_small", kind="global", dim=5, layers=4, bins=8, hidden="32,32", precision="bfloat16",
             exact_inverse=False, chains=20, steps=50, thinning=1),
        # All proposals of one global step of the 64-D mixture run, with their
        # density: the largest flow call.
        dict(name="flow_sample_d64", kind="flow", op="sample_log_prob", dim=64, layers=10, bins=8, hidden="256,256",
             precision="bfloat16", n=409600),
        # Density of a ragged batch through the FP32 conditioner.
        dict(name="flow_log_prob_fp32_d32", kind="flow", op="log_prob", dim=32, layers=8, bins=10, hidden="128,128",
             precision="float32", n=10007),
        # Training steps: the 64-D run's flow, the 32-D flow, and the default
        # bundle's small flow at a small batch.
        dict(name="flow_train_d64", kind="flow_train", dim=64, layers=10, bins=8, hidden="256,256",
             precision="bfloat16", n=10000),
        dict(name="flow_train_d32", kind="flow_train", dim=32, layers=8, bins=10, hidden="128,128",
             precision="bfloat16", n=10000),
        dict(name="flow_train_d5", kind="flow_train", dim=5, layers=4, bins=8, hidden="32,32", precision="bfloat16",
             n=1000),
        # The other model family: RealNVP training step and sampling.
        dict(name="realnvp_train_d32", kind="realnvp_train", dim=32, layers=8, hidden="256", n=10000),
        dict(name="realnvp_sample_d32", kind="realnvp", op="sample", dim=32, layers=8, hidden="256", n=409600),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["local", "local", "batched_hmc", "tempering", "global", "flow", "flow", "flow_train",
                       "flow_train", "realnvp_train", "realnvp"])
    if kind == "local":
        target = rng.choice(["gauss", "rosenbrock", "gmm", "funnel"])
        kernel = rng.choice(["mala", "mala", "grw", "hmc"])
        d = {"gauss": _log_int(rng, 2, 16), "rosenbrock": _log_int(rng, 2, 256), "gmm": _log_int(rng, 2, 128),
             "funnel": _log_int(rng, 2, 256)}[target]
        chains = _log_int(rng, 20, 16384)
        steps = _log_int(rng, 50, 1000)
        # rows kept and work stay below the largest listed case
        steps = max(20, min(steps, int(1.0e8 / (chains * max(d, 8) * (12 if kernel == "hmc" else 1)))))
        return dict(kind=kind, kernel=kernel, target=target, dim=d, chains=chains, steps=steps,
                    thinning=rng.choice([1, 1, 1, 5]),
                    step_size=round(rng.uniform(0.02, 0.1) * (0.2 if target == "rosenbrock" else 1.0), 4))
    if kind == "batched_hmc":
        return dict(kind=kind, targets=rng.randint(4, 32), lo=_log_int(rng, 4, 16), hi=_log_int(rng, 32, 256),
                    chains=_log_int(rng, 20, 400), steps=rng.randint(8, 24), leapfrog=rng.randint(4, 12),
                    step_size=0.05)
    if kind == "tempering":
        d = _log_int(rng, 2, 64)
        return dict(kind=kind, dim=d, modes=rng.randint(2, 8), chains=_log_int(rng, 20, 4096),
                    temps=rng.randint(3, 6), steps=rng.randint(10, 80), step_size=0.05)
    if kind == "global":
        d = _log_int(rng, 2, 32)
        return dict(kind=kind, dim=d, layers=rng.choice([2, 4, 6]), bins=8, hidden=rng.choice(["32,32", "64,64"]),
                    precision=rng.choice(["bfloat16", "bfloat16", "float32"]), exact_inverse=rng.random() < 0.5,
                    chains=_log_int(rng, 20, 1000), steps=_log_int(rng, 10, 100), thinning=rng.choice([1, 1, 5]))
    if kind in ("flow", "flow_train"):
        d = _log_int(rng, 2, 64)
        layers = rng.choice([2, 4, 6, 8, 10])
        h = rng.choice([32, 48, 64, 128, 128, 200, 256])
        c = dict(kind=kind, dim=d, layers=layers, bins=rng.choice([8, 8, 10]),
                 hidden=",".join([str(h)] * rng.choice([1, 2, 2, 2])),
                 precision=rng.choice(["bfloat16", "bfloat16", "float32"]))
        if kind == "flow":
            c["op"] = rng.choice(["log_prob", "sample", "sample_log_prob"])
            c["n"] = _log_int(rng, 20, 200000 if c["precision"] == "bfloat16" else 20000)
        else:
            c["n"] = _log_int(rng, 200, 10000)
        return c
    d = _log_int(rng, 2, 64)
    c = dict(kind=kind, dim=d, layers=rng.choice([2, 4, 8, 10]), hidden=str(rng.choice([32, 64, 100, 128, 256])))
    if kind == "realnvp":
        c["op"] = rng.choice(["log_prob", "sample"])
        c["n"] = _log_int(rng, 20, 200000)
    else:
        c["n"] = _log_int(rng, 200, 10000)
    return c


# ----------------------------------------------------------------- inputs --
def _gen(seed, salt):
    return torch.Generator(device=DEV).manual_seed((int(seed) * 1000003 + salt) & 0x7FFFFFFF)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device=DEV)


def _gauss_params(d, seed):
    g = torch.Generator().manual_seed(int(seed) + 17)
    q, _ = torch.linalg.qr(torch.randn(d, d, generator=g, dtype=F64))
    lam = 10.0 ** (torch.rand(d, generator=g, dtype=F64) * 2 - 1)
    p = q @ torch.diag(1.0 / lam) @ q.T
    return torch.randn(d, generator=g).float(), (0.5 * (p + p.T)).float()


def _gmm_params(d, modes, seed):
    g = torch.Generator().manual_seed(int(seed) + 19)
    means = 4.0 * (torch.randint(0, 2, (modes, d), generator=g).to(F64) * 2 - 1)
    return means, 0.5 + torch.rand(modes, d, generator=g, dtype=F64)


def _target(case, seed):
    """(target, initial positions) as a run past its burn-in meets them."""
    t, d = case.get("target", "gmm"), case["dim"]
    g = _gen(seed, 1)
    n = case["chains"]
    if t == "gauss":
        mean, p = _gauss_params(d, seed)
        return TG.GaussianDense(mean, p), mean.to(DEV) + _randn(g, n, d)
    if t == "rosenbrock":
        return TG.Rosenbrock(d), 1.0 + 0.3 * _randn(g, n, d)
    if t == "funnel":
        return TG.Funnel(d), _randn(g, n, d)
    modes = case.get("modes", 8)
    means, sigmas = _gmm_params(d, modes, seed)
    k = torch.randint(0, modes, (n,), generator=g, device=DEV)
    x = means.to(DEV)[k] + sigmas.to(DEV)[k] * _randn(g, n, d)
    return TG.GaussianMixtureDiag(means, sigmas), x.float()


def _hidden(case):
    return [int(h) for h in case["hidden"].split(",")]


def _spline_theta(case, seed):
    """Flat parameters of a trained-looking spline flow: per layer the scalar
    affine, the conditioner's weights and biases; then the data statistics and
    the N(0, I) base."""
    d, hs, P = case["dim"], _hidden(case), 3 * case["bins"] + 1
    g = _gen(seed, 2)
    parts = []
    ins, outs = [d] + hs, hs + [d * P]
    for _ in range(case["layers"]):
        parts.append(0.1 * _rand(g, 2) - 0.05)
        for i, (a, b) in enumerate(zip(ins, outs)):
            std = (0.3 if i == len(hs) else 0.5) / math.sqrt(a)
            parts.append(std * _randn(g, b * a))
            parts.append((2 * _rand(g, b) - 1) / math.sqrt(a))
    return torch.cat(parts + [_stats(case, seed)])


def _stats(case, seed):
    d = case["dim"]
    g = _gen(seed, 3)
    eye = torch.eye(d, device=DEV)
    var = 0.5 + 3.5 * _rand(g, d)
    return torch.cat([_randn(g, d), torch.diag(var).reshape(-1), torch.zeros(d, device=DEV), eye.reshape(-1)])


def _rnvp_theta(case, seed):
    d, h = case["dim"], _hidden(case)[0]
    g = _gen(seed, 4)
    parts = []
    for _ in range(case["layers"]):
        for _p in range(2):
            parts += [0.5 / math.sqrt(d) * _randn(g, h * d), (2 * _rand(g, h) - 1) / math.sqrt(d),
                      0.3 / math.sqrt(h) * _randn(g, d * h), (2 * _rand(g, d) - 1) / math.sqrt(h) * 0.3]
    return torch.cat(parts + [_stats(case, seed)])


def _flow_data(case, theta, seed):
    """Samples that look like the data the flow was standardised with."""
    d = case["dim"]
    st = theta[-(2 * d + 2 * d * d):]
    sd = torch.sqrt(torch.diagonal(st[d:d + d * d].view(d, d)))
    return st[:d] + sd * _randn(_gen(seed, 5), case["n"], d)


def _adam_moments(n, seed):
    """Moments of a run in progress: gradients of about unit global norm."""
    g = _gen(seed, 6)
    r = 1.0 / math.sqrt(n)
    return 0.3 * r * _randn(g, n), r * r * (0.5 + 1.5 * _rand(g, n))


ADAM = dict(learning_rate=1e-3, b1=0.9, b2=0.999, eps=1e-8, weight_decay=1e-4, max_norm=1.0)
COUNT = 100  # optimiser steps taken before the timed one


def _model(case, seed):
    if case["kind"].startswith("realnvp"):
        m = RealNVP(case["dim"], case["layers"], _hidden(case)[0], fr.PRNGKey(seed))
        m.theta.copy_(_rnvp_theta(case, seed))
    else:
        m = MaskedCouplingRQSpline(case["dim"], case["layers"], _hidden(case), case["bins"], fr.PRNGKey(seed),
                                   precision=case["precision"],
                                   exact_inverse=case.get("exact_inverse", case.get("op") == "sample_log_prob"))
        m.theta.copy_(_spline_theta(case, seed))
    m.mark_updated()
    return m


def _step_buffers(case):
    rows = (case["steps"] + case["thinning"] - 1) // case["thinning"]
    return {"pos": Buffer("pos", (case["chains"], rows, case["dim"]), 1),
            "lp": Buffer("lp", (case["chains"], rows), 1),
            "acc": Buffer("acc", (case["chains"], rows), 1),
            "state": State({"p": "pos", "l": "lp", "a": "acc"}, name="state")}


def _funnel_dims(case):
    n = case["targets"]
    r = math.log(case["hi"] / case["lo"])
    return [int(round(case["lo"] * math.exp(r * ((7 * i) % n) / max(1, n - 1)))) for i in range(n)]


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, "key": fr.PRNGKey(seed)}
    if kind == "local":
        tgt, x = _target(case, seed)
        kernel = {"mala": MALA, "grw": GaussianRandomWalk}.get(case["kernel"])
        kernel = kernel(case["step_size"]) if kernel else HMC(step_size=case["step_size"], n_leapfrog=10)
        s["res"] = dict(_step_buffers(case), logpdf=LogPDF(tgt, n_dims=case["dim"]), kernel=kernel)
        s["strategy"] = TakeSerialSteps("logpdf", "kernel", "state", ["p", "l", "a"], case["steps"],
                                        thinning=case["thinning"])
        s["x"] = x
    elif kind == "batched_hmc":
        dims, c, t = _funnel_dims(case), case["chains"], case["steps"]
        bh = BatchedHMC([TG.Funnel(d) for d in dims], c, step_size=case["step_size"], n_leapfrog=case["leapfrog"])
        for i, x in enumerate(bh.x):
            x.copy_(_randn(_gen(seed, 100 + i), c, dims[i]))
        outs = [tuple(torch.zeros(sh, device=DEV) for sh in ((c, t, d), (c, t), (c, t))) + (0,) for d in dims]
        s.update(bh=bh, outs=outs, launch=bh.prepare(s["key"], t, outputs=outs))
    elif kind == "tempering":
        tgt, x = _target(case, seed)
        n, t, d = case["chains"], case["temps"], case["dim"]
        temps = Buffer("temperature", (t,), 0)
        temps.update_buffer(torch.linspace(1.0, 5.0, t))
        tpos = Buffer("tempered_positions", (n, t - 1, d), 2)
        tpos.update_buffer(x[:, None].expand(n, t - 1, d))
        s["res"] = {"tlp": TemperedPDF(LogPDF(tgt, n_dims=d), None, n_dims=d, n_temps=t),
                    "mala": MALA(case["step_size"], fused_steps=case["steps"]), "tp": tpos, "T": temps,
                    "state": State({"training": True}, name="sampler_state")}
        s["strategy"] = ParallelTempering(case["steps"], "tlp", "mala", ["tp", "T"], "state")
        s["x"] = x
    elif kind == "global":
        tgt, x = _target(case, seed)
        s["res"] = dict(_step_buffers(case), logpdf=LogPDF(tgt, n_dims=case["dim"]),
                        kernel=NFProposal(_model(case, seed)))
        s["strategy"] = TakeGroupSteps("logpdf", "kernel", "state", ["p", "l", "a"], case["steps"],
                                       thinning=case["thinning"])
        s["x"] = x
    else:
        s["model"] = m = _model(case, seed)
        if kind.endswith("train"):
            mu, nu = _adam_moments(m.theta.numel(), seed)
            s.update(x=_flow_data(case, m.theta, seed), optim=AdamWClip(**ADAM), opt_state=AdamState(mu, nu, COUNT))
        elif case["op"] == "log_prob":
            s["x"] = _flow_data(case, m.theta, seed)
    return s


# -------------------------------------------------------------------- run --
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind in ("local", "global"):
        _, res, last = s["strategy"](s["key"], s["res"], s["x"], {})
        return {"last": last, "pos": res["pos"].data, "lp": res["lp"].data, "acc": res["acc"].data}
    if kind == "batched_hmc":
        s["launch"]()
        return {"pos": [o[0] for o in s["outs"]], "lp": [o[1] for o in s["outs"]]}
    if kind == "tempering":
        _, res, x = s["strategy"](s["key"], s["res"], s["x"], {})
        return {"x": x, "tempered": res["tp"].data, "temps": res["T"].data}
    m = s["model"]
    if kind.endswith("train"):
        loss, m, st = m.train_step(s["x"], s["optim"], s["opt_state"])
        return {"loss": loss, "theta": m.theta, "mu": st.mu, "nu": st.nu}
    if case["op"] == "log_prob":
        return m.log_prob(s["x"])
    if case["op"] == "sample":
        return m.sample(s["key"], case["n"])
    return m.sample_and_log_prob(s["key"], case["n"])


# ------------------------------------------------------------------- work --
def _target_flops(case):
    d = case["dim"]
    return {"gauss": 2 * d * d + 4 * d, "rosenbrock": 14 * d, "funnel": 4 * d, "gmm": 7 * d * case.get("modes", 8)}[
        case.get("target", "gmm")]


def _flow_macs(case):
    """(conditioner multiply-adds, transformed dims) a sample over all layers."""
    d, P = case["dim"], (3 * case["bins"] + 1) if "bins" in case else 2
    hs, macs, tr = _hidden(case), 0, 0
    for l in range(case["layers"]):
        dc = (d + 1) // 2 if l % 2 else d // 2
        m = dc * hs[0] + sum(a * b for a, b in zip(hs, hs[1:]))
        macs += (2 * (dc * hs[0] + hs[0] * (d - dc))) if "bins" not in case else m + hs[-1] * (d - dc) * P
        tr += d - dc
    return macs, tr


def _n_theta(case):
    d, hs = case["dim"], _hidden(case)
    if "bins" not in case:
        return case["layers"] * 2 * (2 * hs[0] * d + hs[0] + d) + 2 * d + 2 * d * d
    ins, outs = [d] + hs, hs + [d * (3 * case["bins"] + 1)]
    return case["layers"] * (2 + sum(b * (a + 1) for a, b in zip(ins, outs))) + 2 * d + 2 * d * d


def work(case):
    kind, d = case["kind"], case["dim"] if "dim" in case else 0
    if kind in ("local", "tempering"):
        rows = case["chains"] * case.get("temps", 1)
        kept = 0 if kind == "tempering" else (case["steps"] + case["thinning"] - 1) // case["thinning"]
        per = _target_flops(case) + 12 * d + 15 * d  # value and gradient, proposal and ratio, normals
        if case.get("kernel") == "hmc":
            per = 11 * (_target_flops(case) + 4 * d) + 21 * d
        return {"bytes": 4.0 * rows * (2 * d + kept * (d + 2)), "flops": float(rows * case["steps"] * per)}
    if kind == "batched_hmc":
        n, L, sd = case["chains"], case["leapfrog"], sum(_funnel_dims(case))
        nt = case["targets"]
        return {"bytes": 4.0 * n * (2 * sd + case["steps"] * (sd + 2 * nt)),
                "flops": float(n * case["steps"] * sd * (7 * (L + 1) + 24))}
    n = case["chains"] * case["steps"] if kind == "global" else case["n"]
    macs, tr = _flow_macs(case)
    spline = 120 if "bins" in case else 8
    th = 4.0 * _n_theta(case)
    if kind == "global":
        rows = case["chains"] * ((case["steps"] + case["thinning"] - 1) // case["thinning"])
        passes = n * (1 if case["exact_inverse"] else 2) + case["chains"]
        return {"bytes": th + 4.0 * (rows * (d + 2) + 2 * case["chains"] * d),
                "flops": float(passes * (2 * macs + spline * tr) + n * _target_flops(case))}
    if kind.endswith("train"):
        return {"bytes": 6 * th + 4.0 * n * d, "flops": float(n * (6 * macs + 3 * spline * tr))}
    return {"bytes": th + 4.0 * n * (d + (case["op"] == "sample_log_prob")) + (4.0 * n if case["op"] == "log_prob" else 0),
            "flops": float(n * (2 * macs + spline * tr))}


# -------------------------------------------------- FP64: random numbers --
M32 = 0xFFFFFFFF


def _philox(c0, c1, c2, c3, key):
    """Philox4x32-10 on int64 tensors holding 32-bit words (the wrapped 64-bit
    product has the right bits: its high word is masked after the shift)."""
    k0, k1 = int(key[0]), int(key[1])
    for _ in range(10):
        p0, p1 = c0 * 0xD2511F53, c2 * 0xCD9E8D57
        c0, c1, c2, c3 = ((p1 >> 32) & M32) ^ c1 ^ k0, p1 & M32, ((p0 >> 32) & M32) ^ c3 ^ k1, p0 & M32
        k0, k1 = (k0 + 0x9E3779B9) & M32, (k1 + 0xBB67AE85) & M32
    return c0, c1, c2, c3


def _u01(w):
    return ((w >> 9).to(F64) + 0.5) * 2.0 ** -23


def _normals(key, rows, d, step, sid):
    """[rows, d] standard normals of one step: Box-Muller on 4-word blocks."""
    ch = (d + 3) // 4
    c0 = torch.arange(ch, device=DEV)[None, :].expand(rows, ch)
    c1 = torch.arange(rows, device=DEV)[:, None].expand(rows, ch)
    w = _philox(c0, c1, torch.full_like(c0, step), torch.full_like(c0, sid), key)
    r0, r1 = (torch.sqrt(-2 * torch.log(_u01(v))) for v in (w[0], w[2]))
    a0, a1 = (2 * math.pi * _u01(v) for v in (w[1], w[3]))
    z = torch.stack([r0 * torch.cos(a0), r0 * torch.sin(a0), r1 * torch.cos(a1), r1 * torch.sin(a1)], -1)
    return z.reshape(rows, 4 * ch)[:, :d]


def _log_u(key, rows, step, sid):
    c1 = torch.arange(rows, device=DEV)
    w = _philox(torch.zeros_like(c1), c1, torch.full_like(c1, step), torch.full_like(c1, sid), key)
    return torch.log(_u01(w[0]))


def _words(*ctr, key):
    return [int(v) for v in _philox(*(torch.tensor(c) for c in ctr), key)]


SPLIT = 0x53504C54


def _child(key, i):
    return _words(i, 0, 0, SPLIT, key=key)[:2]


def _root(seed):
    return [(int(seed) >> 32) & M32, int(seed) & M32]


def _f32(v):
    return float(np.float32(v))


# ------------------------------------------------------- FP64: densities --
def _density(case, seed):
    """x -> (log p, gradient) in FP64, on the FP32 parameters of the target."""
    t, d = case.get("target", "gmm"), case["dim"]
    if t == "gauss":
        mean, p = (v.to(DEV, F64) for v in _gauss_params(d, seed))

        def f(x):
            y = x - mean
            g = -(y @ p)
            return 0.5 * (y * g).sum(-1), g
    elif t == "rosenbrock":
        sc = _f32(1.0 / 20.0)

        def f(x):
            a, b = x[:, :-1], x[:, 1:]
            r, o = b - a * a, 1 - a
            g = torch.zeros_like(x)
            g[:, :-1] += -400 * a * r - 2 * o
            g[:, 1:] += 200 * r
            return -sc * (100 * r * r + o * o).sum(-1), -sc * g
    elif t == "funnel":
        f = _funnel
    else:
        means, sigmas = _gmm_params(d, case.get("modes", 8), seed)
        K = means.shape[0]
        c = (torch.log(torch.full((K,), 1.0 / K, dtype=F64)) - torch.log(sigmas).sum(-1)).float().to(DEV, F64)
        mu, isg = means.float().to(DEV, F64), (1 / sigmas).float().to(DEV, F64)

        def f(x):
            q = torch.stack([c[k] - 0.5 * (((x - mu[k]) * isg[k]) ** 2).sum(-1) for k in range(K)], -1)
            w = torch.softmax(q, -1)
            g = torch.zeros_like(x)
            for k in range(K):
                g -= w[:, k:k + 1] * (x - mu[k]) * isg[k] ** 2
            return torch.logsumexp(q, -1), g
    return f


def _funnel(x):
    v, y = x[:, 0], x[:, 1:]
    em, s, n = torch.exp(-v), (y * y).sum(-1), x.shape[1] - 1
    g = torch.cat([(-v / 9 - 0.5 * n + 0.5 * em * s)[:, None], -y * em[:, None]], 1)
    return -v * v / 18 - 0.5 * n * v - 0.5 * em * s, g


# ---------------------------------------------------------- FP64: chains --
def _chain(kernel, f, x, key, steps, dt, leapfrog=10, keep=None):
    """``steps`` Metropolis steps of every row; keep(step, x, logp, accept)."""
    lp, g = f(x)
    n, d = x.shape
    for s in range(steps):
        if kernel == "hmc":
            p = _normals(key, n, d, s, 2)
            h0 = -lp + 0.5 * (p * p).sum(-1)
            p, y, gy = p + 0.5 * dt * g, x, g
            for i in range(leapfrog + 1):
                y = y + dt * p
                ly, gy = f(y)
                p = p + (dt if i < leapfrog else 0.5 * dt) * gy
            ratio, lu = h0 - (-ly + 0.5 * (p * p).sum(-1)), _log_u(key, n, s, 3)
        else:
            z = _normals(key, n, d, s, 0 if kernel == "mala" else 7)
            h = 0.5 * dt * dt if kernel == "mala" else 0.0
            y = x + h * g + dt * z
            ly, gy = f(y)
            ratio = ly - lp
            if kernel == "mala":
                ratio = ratio + ((dt * z) ** 2 - (x - y - h * gy) ** 2).sum(-1) / (2 * dt * dt)
            lu = _log_u(key, n, s, 1 if kernel == "mala" else 8)
        acc = lu < ratio
        x, g, lp = torch.where(acc[:, None], y, x), torch.where(acc[:, None], gy, g), torch.where(acc, ly, lp)
        if keep:
            keep(s, x, lp, acc)
    return x


def _exact_local(case, seed):
    _, x = _target(case, seed)
    key = _child(_root(seed), 1)
    n, d, th = case["chains"], case["dim"], case["thinning"]
    rows = (case["steps"] + th - 1) // th
    pos = torch.zeros(n, rows, d, device=DEV, dtype=F64)
    lps, accs = torch.zeros(n, rows, device=DEV, dtype=F64), torch.zeros(n, rows, device=DEV, dtype=F64)

    def keep(s, x, lp, acc):
        if s % th == 0:
            pos[:, s // th], lps[:, s // th], accs[:, s // th] = x, lp, acc.to(F64)

    last = _chain(case["kernel"], _density(case, seed), x.to(F64), key, (rows - 1) * th + 1, _f32(case["step_size"]),
                  keep=keep)
    return {"last": last, "pos": pos, "lp": lps, "acc": accs}


def _exact_batched_hmc(case, seed):
    poss, lpss = [], []
    for i, d in enumerate(_funnel_dims(case)):
        n, t = case["chains"], case["steps"]
        x = _randn(_gen(seed, 100 + i), n, d).to(F64)
        key = _words(i, 0, 1, SPLIT, key=_root(seed))[:2]
        pos, lps = torch.zeros(n, t, d, device=DEV, dtype=F64), torch.zeros(n, t, device=DEV, dtype=F64)

        def keep(s, y, lp, acc, pos=pos, lps=lps):
            pos[:, s], lps[:, s] = y, lp

        _chain("hmc", _funnel, x, key, t, _f32(case["step_size"]), case["leapfrog"], keep)
        poss.append(pos)
        lpss.append(lps)
    return {"pos": poss, "lp": lpss}


def _exact_tempering(case, seed):
    n, T, d = case["chains"], case["temps"], case["dim"]
    _, x0 = _target(case, seed)
    f = _density(case, seed)
    temps = torch.linspace(1.0, 5.0, T).to(DEV, F64)
    beta = (1 / temps).repeat(n)
    k1 = _child(_root(seed), 0)  # the strategy splits its key once before the steps and once before the swaps
    steps_key, k2 = _child(k1, 1), _child(k1, 0)
    swap_key = _child(k2, 1)

    def tempered(x):
        lp, g = f(x)
        return beta * lp, beta[:, None] * g

    x = x0.to(F64)[:, None].expand(n, T, d).reshape(n * T, d)
    x = _chain("mala", tempered, x, steps_key, case["steps"], _f32(case["step_size"]))
    ll = f(x)[0].reshape(n, T)
    x = x.reshape(n, T, d)
    rows = torch.arange(n, device=DEV)
    out, cur, lc = x.clone(), torch.zeros(n, dtype=torch.int64, device=DEV), ll[:, 0]
    rate = []
    for i in range(T - 1):
        w = _philox(torch.zeros_like(rows), rows, torch.full_like(rows, i), torch.full_like(rows, 9), swap_key)
        a = torch.log(_u01(w[0])) < (1 / temps[i + 1] - 1 / temps[i]) * (lc - ll[:, i + 1])
        out[:, i] = torch.where(a[:, None], x[:, i + 1], x[rows, cur])
        cur = torch.where(a, cur, torch.full_like(cur, i + 1))
        lc = torch.where(a, lc, ll[:, i + 1])
        rate.append(a.to(F64).mean())
    out[:, T - 1] = x[rows, cur]
    new = temps.clone()
    for i in range(1, T - 1):
        new[i] = new[i - 1] + (temps[i] - temps[i - 1]) * torch.exp(100.0 / n * (rate[i - 1] - rate[i]))
    return {"x": out[:, 0], "tempered": out[:, 1:], "temps": new}


# ----------------------------------------------------------- FP64: flows --
def _spline_knots(raw, K):
    lo, hi, mn = -10.0, 10.0, _f32(1e-4)
    w = torch.softmax(raw[..., :K], -1) * (hi - lo - K * mn) + mn
    h = torch.softmax(raw[..., K:2 * K], -1) * (hi - lo - K * mn) + mn
    off = math.log(math.exp(1.0 - mn) - 1.0)
    s = torch.nn.functional.softplus(raw[..., 2 * K:] + off) + mn

    def knots(b):
        c = lo + torch.cumsum(b[..., :-1], -1)
        return torch.cat([torch.full_like(b[..., :1], lo), c, torch.full_like(b[..., :1], hi)], -1)

    return knots(w), knots(h), s


def _spline(v, raw, K, inverse):
    """Rational-quadratic spline of v: (value, log-derivative)."""
    xp, yp, s = _spline_knots(raw, K)
    ref = yp if inverse else xp
    below, above = v <= -10.0, v >= 10.0
    vc = v.clamp(-10.0 + 1e-9, 10.0 - 1e-9)
    k = (torch.searchsorted(ref.detach().contiguous(), vc.detach()[..., None].contiguous(), right=True) - 1).clamp(0, K - 1)

    def at(a, i):
        return torch.gather(a, -1, i)[..., 0]

    xk, xk1, yk, yk1 = at(xp, k), at(xp, k + 1), at(yp, k), at(yp, k + 1)
    dk, dk1 = at(s, k), at(s, k + 1)
    w, h = xk1 - xk, yk1 - yk
    r = h / w
    st = dk1 + dk - 2 * r
    if inverse:
        q = ((vc - yk) / h).clamp(0, 1)
        c, b = -r * q, dk - st * q
        sq = torch.sqrt((b * b - 4 * (r - b) * c).clamp_min(0))
        z = torch.where(b >= 0, 2 * c / torch.where(b >= 0, -b - sq, torch.ones_like(b)),
                        (-b + sq) / torch.where(b >= 0, torch.ones_like(b), 2 * (r - b))).clamp(0, 1)
    else:
        z = ((vc - xk) / w).clamp(0, 1)
    zz = z * (1 - z)
    den = r + st * zz
    ld = 2 * torch.log(r) + torch.log(dk1 * z * z + 2 * r * zz + dk * (1 - z) ** 2) - 2 * torch.log(den)
    out = w * z + xk if inverse else yk + h * (r * z * z + dk * zz) / den
    edge, se = torch.where(below, torch.full_like(v, -10.0), torch.full_like(v, 10.0)), torch.where(below, s[..., 0], s[..., -1])
    lin = (v - edge) / se + edge if inverse else (v - edge) * se + edge
    tail = below | above
    ld = torch.where(tail, torch.log(se), ld)
    return torch.where(tail, lin, out), -ld if inverse else ld


def _spline_layers(case, th):
    d, hs, P = case["dim"], _hidden(case), 3 * case["bins"] + 1
    ins, outs = [d] + hs, hs + [d * P]
    o, layers = 0, []
    for _ in range(case["layers"]):
        lay = {"sc": th[o], "sh": th[o + 1], "lin": []}
        o += 2
        for a, b in zip(ins, outs):
            lay["lin"].append((th[o:o + a * b].view(b, a), th[o + a * b:o + a * b + b]))
            o += a * b + b
        layers.append(lay)
    return layers


def _spline_map(case, layers, x, direction):
    """forward, or inverse in the reference's layer order ("ref") or exactly ("exact")."""
    d, K = case["dim"], case["bins"]
    P = 3 * K + 1
    ld = torch.zeros(x.shape[0], device=x.device, dtype=x.dtype)
    for l in (range(len(layers)) if direction == "forward" else reversed(range(len(layers)))):
        lay = layers[l]
        ct = [j for j in range(d) if (j + l) % 2 == 1], [j for j in range(d) if (j + l) % 2 == 0]
        sc, sh = lay["sc"], lay["sh"]
        if direction == "forward":
            x, ld = (x + sh) * torch.exp(sc), ld + d * sc
        elif direction == "ref":
            x, ld = x * torch.exp(-sc) - sh, ld - d * sc
        h = x[:, ct[0]]
        for i, (w, b) in enumerate(lay["lin"]):
            if i == len(lay["lin"]) - 1:
                rows = (torch.tensor(ct[1], device=x.device)[:, None] * P + torch.arange(P, device=x.device)).reshape(-1)
                h = (h @ w[rows].T + b[rows]).view(-1, len(ct[1]), P)
            else:
                h = torch.tanh(h @ (w[:, ct[0]] if i == 0 else w).T + b)
        y, l1 = _spline(x[:, ct[1]].contiguous(), h, K, direction != "forward")
        x, ld = x.index_copy(1, torch.tensor(ct[1], device=x.device), y), ld + l1.sum(-1)
        if direction == "exact":
            x, ld = x * torch.exp(-sc) - sh, ld - d * sc
    return x, ld


def _rnvp_map(case, th, x, inverse):
    d, h = case["dim"], _hidden(case)[0]
    sz = 2 * h * d + h + d
    ld = torch.zeros(x.shape[0], device=x.device, dtype=x.dtype)
    for l in (reversed(range(case["layers"])) if inverse else range(case["layers"])):
        first, rest = list(range(d // 2)), list(range(d // 2, d))
        c, t = (first, rest) if l % 2 == 0 else (rest, first)
        outs = []
        for p in range(2):
            o = (2 * l + p) * sz
            w1, b1 = th[o:o + h * d].view(h, d), th[o + h * d:o + h * d + h]
            o += h * d + h
            w2, b2 = th[o:o + d * h].view(d, h), th[o + d * h:o + d * h + d]
            outs.append(torch.relu(x[:, c] @ w1[:, c].T + b1) @ w2[t].T + b2[t])
        s, sh = torch.tanh(outs[0]), outs[1]
        y = x[:, t] * torch.exp(-s) - sh if inverse else (x[:, t] + sh) * torch.exp(s)
        x, ld = x.index_copy(1, torch.tensor(t, device=x.device), y), ld + (-s if inverse else s).sum(-1)
    return x, ld


def _map(case, th, x, direction):
    if "bins" not in case:
        return _rnvp_map(case, th, x, direction != "forward")
    return _spline_map(case, _spline_layers(case, th), x, direction)


def _chunks(n, d):
    step = max(256, min(n, (1 << 21) // max(8, d)))
    return [(a, min(n, a + step)) for a in range(0, n, step)]


def _exact_log_prob(case, th, x):
    d = case["dim"]
    st = th[-(2 * d + 2 * d * d):]
    z = (x - st[:d]) / torch.sqrt(torch.diagonal(st[d:d + d * d].view(d, d)))
    y, ld = _map(case, th, z, "forward")
    return ld - 0.5 * (y * y).sum(-1) - 0.5 * d * math.log(2 * math.pi)


def _exact_sample(case, th, z, direction):
    d = case["dim"]
    st = th[-(2 * d + 2 * d * d):]
    x, ld = _map(case, th, z, direction)
    x = x * torch.sqrt(torch.diagonal(st[d:d + d * d].view(d, d))) + st[:d]
    return x, -0.5 * (z * z).sum(-1) - 0.5 * d * math.log(2 * math.pi) - ld


def _theta(case, seed):
    return (_spline_theta if "bins" in case else _rnvp_theta)(case, seed).to(F64)


def _exact_flow(case, seed):
    th, n, d = _theta(case, seed), case["n"], case["dim"]
    if case["op"] == "log_prob":
        x = _flow_data(case, th.float(), seed).to(F64)
        return torch.cat([_exact_log_prob(case, th, x[a:b]) for a, b in _chunks(n, d)])
    z = _normals(_root(seed), n, d, 0, 5)
    got = [_exact_sample(case, th, z[a:b], "exact" if case["op"] == "sample_log_prob" else "ref")
           for a, b in _chunks(n, d)]
    x = torch.cat([v[0] for v in got])
    return x if case["op"] == "sample" else (x, torch.cat([v[1] for v in got]))


def _exact_train(case, seed):
    th, n, d = _theta(case, seed), case["n"], case["dim"]
    x = _flow_data(case, th.float(), seed).to(F64)
    grad, loss = torch.zeros_like(th), 0.0
    n_w = th.numel() - 2 * d - 2 * d * d
    for a, b in _chunks(n, 16 * d):
        p = th[:n_w].clone().requires_grad_(True)
        part = -_exact_log_prob(case, torch.cat([p, th[n_w:]]), x[a:b]).sum() / n
        grad[:n_w] += torch.autograd.grad(part, p)[0]
        loss = loss + part.detach()
    norm = torch.linalg.norm(grad)
    u = torch.where(norm < ADAM["max_norm"], grad, grad / norm * ADAM["max_norm"])
    mu, nu = (v.to(F64) for v in _adam_moments(th.numel(), seed))
    b1, b2, t = _f32(ADAM["b1"]), _f32(ADAM["b2"]), COUNT + 1
    mu, nu = b1 * mu + (1 - b1) * u, b2 * nu + (1 - b2) * u * u
    step = mu / (1 - b1 ** t) / (torch.sqrt(nu / (1 - b2 ** t)) + ADAM["eps"]) + ADAM["weight_decay"] * th
    return {"loss": loss, "theta": th - ADAM["learning_rate"] * step, "mu": mu, "nu": nu}


def _exact_global(case, seed):
    """The Metropolis-Hastings scan over the flow's proposals. With the BF16
    conditioner the proposals' densities carry its rounding, which decides
    some steps: no exact rows there."""
    if case["precision"] != "float32":
        return None
    n, S, d, th = case["chains"], case["steps"], case["dim"], case["thinning"]
    _, x0 = _target(case, seed)
    x0 = x0.to(F64)
    p, key = _theta(case, seed), _child(_root(seed), 1)
    z = _normals(key, n * S, d, 0, 5)
    prop, q = _exact_sample(case, p, z, "exact" if case["exact_inverse"] else "ref")
    if not case["exact_inverse"]:
        q = _exact_log_prob(case, p, prop)
    f = _density(case, seed)
    prop, q, lpp = prop.view(n, S, d), q.view(n, S), f(prop)[0].view(n, S)
    x, qc, lp = x0, _exact_log_prob(case, p, x0), f(x0)[0]
    pos, lps, accs = [], [], []
    for s in range(S):
        acc = _log_u(key, n, s, 4) < (lpp[:, s] - lp) - (q[:, s] - qc)
        x = torch.where(acc[:, None], prop[:, s], x)
        qc, lp = torch.where(acc, q[:, s], qc), torch.where(acc, lpp[:, s], lp)
        if s % th == 0:
            pos.append(x)
            lps.append(lp)
            accs.append(acc.to(F64))
    return {"last": pos[-1], "pos": torch.stack(pos, 1), "lp": torch.stack(lps, 1), "acc": torch.stack(accs, 1)}


def exact(case, seed):
    return {"local": _exact_local, "batched_hmc": _exact_batched_hmc, "tempering": _exact_tempering,
            "global": _exact_global, "flow": _exact_flow, "realnvp": _exact_flow, "flow_train": _exact_train,
            "realnvp_train": _exact_train}[case["kind"]](case, seed)
