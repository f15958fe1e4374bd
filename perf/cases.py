"""Performance cases: what users of this library have it do, through its public entry points.

A case names an entry point and the sizes, types and options of one call:

  entry "select"   ggms.select: device vector, ranks and results on the host (the reference's call shape)
  entry "topk"     ggms.topk: the K largest values
  entry "device"   ggms.select_device with the device-driven schedule: ranks and results stay on the device
  entry "batch"    ggms.batch.BatchPlan, replayed as a hipGraph with the committed autotuner table
  entry "train"    one training step of the learned splitter's network (loss and gradient, then Adam)

The inputs come from torch and numpy generators seeded by `seed` alone.
"""
import ctypes
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ggms-distributed_amd"))
import ggms  # noqa: E402
from ggms import autotune, learned  # noqa: E402
from ggms.batch import BatchPlan  # noqa: E402

DEV = "cuda:0"
TORCH = {"float32": torch.float32, "float64": torch.float64, "uint32": torch.uint32, "int32": torch.int32}
SIZE = {"float32": 4, "float64": 8, "uint32": 4, "int32": 4}


def _select(name, dtype, dist, n, nk, kdist, **kw):
    return dict({"name": name, "entry": "select", "dtype": dtype, "dist": dist, "n": n, "nk": nk, "kdist": kdist,
                 "alg": "iterative", "splitter": "linear", "offset": 0}, **kw)


def listed():
    return [
        # a summary (the deciles) of a short vector: launches and latency only
        _select("deciles_1k_f32", "float32", "normal", 1000, 9, "even"),
        # a serving loop's call: integer keys, ranks and results resident, nothing read back between kernels
        _select("device_100k_i32", "int32", "full_range", 100_003, 32, "uniform_random", entry="device"),
        # one-pass selection of 101 sorted distinct ranks of a mid-sized uniform vector
        _select("bucket_1m_uniform_f32", "float32", "uniform", 1 << 20, 101, "distinct_sorted", alg="bucket"),
        # the 1024 largest of a slice of a longer, long-tailed score vector (its base is 4-byte aligned only)
        _select("topk_10m_f32", "float32", "lognormal", 10_000_019, 1024, "top", entry="topk", alg="bucket", offset=1),
        # the benchmark's workload: many ranks of a whole-GPU vector
        _select("normal_2p28_f32", "float32", "normal", 1 << 28, 1001, "uniform_random"),
        # the same in double precision
        _select("normal_2p27_f64", "float64", "normal", 1 << 27, 1001, "uniform_random"),
        # heavy duplicates: every value occurs tens of thousands of times
        _select("dups_2p26_u32", "uint32", "mod_1024", 1 << 26, 8192, "even"),
        # a fine quantile grid of one-sided data
        _select("halfnormal_2p26_f32", "float32", "half_normal", 1 << 26, 8192, "even"),
        # one value holds 99 % of the vector (a sparse feature), a fine quantile grid
        _select("constant99_2p26_f32", "float32", "near_constant", 1 << 26, 8192, "even"),
        # multi-modal data, thousands of ranks, the trained splitter
        _select("mixture_2p28_learned", "float32", "mixture", 1 << 28, 8192, "uniform_random", splitter="learned"),
        # thousands of independent problems of uneven sizes in one launch
        {"name": "batch_4096", "entry": "batch", "dtype": "float32", "problems": 4096, "log2_lo": 10, "log2_hi": 22,
         "max_ks": 512},
        # one step of the splitter network's training loop at its default batch
        {"name": "train_4096", "entry": "train", "nb": 4096},
    ]


def draw(rng: random.Random):
    u = rng.random()
    if u < 0.12:
        lo = rng.randint(8, 14)
        hi = rng.randint(lo + 2, 22)
        problems = int(2 ** rng.uniform(6, 12))
        return {"entry": "batch", "dtype": rng.choice(["float32", "float32", "float64", "uint32"]),
                "problems": min(problems, (1 << 32) >> hi), "log2_lo": lo, "log2_hi": hi,
                "max_ks": int(2 ** rng.uniform(0, 9))}
    if u < 0.2:
        return {"entry": "train", "nb": int(2 ** rng.uniform(8, 16))}
    dtype = rng.choice(["float32", "float32", "float64", "uint32", "int32"])
    if dtype in ("uint32", "int32"):
        dist = rng.choice(["full_range", "full_range", "mod_1024"])
    else:
        dist = rng.choice(["uniform", "normal", "normal", "half_normal", "lognormal", "mixture", "near_constant"])
    n = int(2 ** rng.uniform(9, 27 if dtype == "float64" else 28))
    nk = max(1, min(n, int(2 ** rng.uniform(0, 13))))
    case = {"entry": "select", "dtype": dtype, "dist": dist, "n": n, "nk": nk,
            "kdist": rng.choice(["uniform_random", "uniform_random", "distinct_sorted", "even", "window"]),
            "alg": rng.choice(["iterative", "iterative", "bucket", "distributed", "distributed_bucket"]),
            "splitter": rng.choice(["linear", "linear", "learned", "sketch"]), "offset": rng.choice([0, 0, 0, 1])}
    if case["alg"].startswith("distributed"):
        case["splitter"] = "linear"
    v = rng.random()
    if v < 0.15:
        case.update(entry="topk", kdist="top", nk=min(nk, 2048))
    elif v < 0.3:
        case.update(entry="device", splitter="linear")
    return case


def _seeds(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g, np.random.default_rng(int(seed))


def _values(dtype, dist, n, g, rng):
    """n values of a distribution, on the device."""
    if dtype in ("uint32", "int32"):
        if dist == "mod_1024":
            v = torch.randint(0, 1024, (n,), dtype=torch.int32, device=DEV, generator=g)
        else:
            v = torch.empty(n, dtype=torch.int32, device=DEV)
            v.random_(-(1 << 31), 1 << 31, generator=g)
        return v.view(torch.uint32) if dtype == "uint32" else v
    x = torch.empty(n, dtype=TORCH[dtype], device=DEV)
    if dist == "uniform":
        return x.uniform_(0, 1, generator=g)
    if dist == "lognormal":
        return x.log_normal_(0, 1, generator=g)
    x.normal_(0, 1, generator=g)
    if dist == "half_normal":
        x.abs_()
    elif dist == "near_constant":
        keep = torch.empty(n, dtype=torch.float32, device=DEV).uniform_(0, 1, generator=g) < 0.01
        x.masked_fill_(~keep, float(np.float32(rng.standard_normal())))
    elif dist == "mixture":  # 1 to 8 Gaussians beside a lognormal tail
        m = int(rng.integers(1, 9))
        mu, sg = rng.uniform(-100, 100, m), 10.0 ** rng.uniform(-2, 1, m)
        tail = torch.empty(n, dtype=torch.float32, device=DEV).uniform_(0, 1, generator=g)
        which = torch.empty(n, dtype=torch.int8, device=DEV).random_(0, m, generator=g)
        y = x.exp()
        for c in range(m):
            at = (which == c) & (tail >= 0.05)
            y = torch.where(at, x * float(sg[c]) + float(mu[c]), y)
        x = y
    return x


def _ranks(kdist, nk, n, rng):
    if kdist == "top":
        ks = np.arange(1, nk + 1)
    elif kdist == "even":
        ks = -(-np.arange(1, nk + 1, dtype=np.int64) * n // nk)
    elif kdist == "window":
        w = min(n, max(nk, n // 100))
        ks = int(rng.integers(0, n - w + 1)) + rng.integers(1, w + 1, nk)
    elif kdist == "distinct_sorted":
        ks = rng.integers(1, n + 1, nk) if n > 1 << 24 else rng.choice(n, nk, replace=False) + 1
        ks = np.unique(ks)
        while len(ks) < nk:
            ks = np.unique(np.concatenate([ks, rng.integers(1, n + 1, nk - len(ks))]))
    else:
        ks = rng.integers(1, n + 1, nk)
    return np.clip(ks, 1, n).astype(np.uint32)


def _select_inputs(case, seed):
    g, rng = _seeds(seed)
    off = case["offset"]
    x = _values(case["dtype"], case["dist"], case["n"] + off, g, rng)[off:]
    return x, _ranks(case["kdist"], case["nk"], case["n"], rng)


def _batch_inputs(case, seed):
    g, rng = _seeds(seed)
    p = case["problems"]
    sizes = np.clip(np.floor(2.0 ** rng.uniform(case["log2_lo"], case["log2_hi"], p)), 1, None).astype(np.int64)
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint64)
    nks = np.random.default_rng(p).integers(1, case["max_ks"] + 1, p)  # the batch's shape: the same for every seed
    koff = np.concatenate([[0], np.cumsum(nks)]).astype(np.uint32)
    ks = np.concatenate([rng.integers(1, s + 1, k) for s, k in zip(sizes, nks)]).astype(np.uint32)
    which = rng.integers(0, 3, p)
    if case["dtype"] == "uint32":
        x = _values("uint32", "full_range", int(off[-1]), g, rng)
    else:  # each problem uniform, normal or lognormal
        x = torch.empty(int(off[-1]), dtype=TORCH[case["dtype"]], device=DEV).normal_(0, 1, generator=g)
        for i in range(p):
            v = x[int(off[i]):int(off[i + 1])]
            if which[i] == 0:
                v.uniform_(0, 1, generator=g)
            elif which[i] == 1:
                v.exp_()
    return x, off, ks, koff


def _train_inputs(case, seed):
    """A batch of sorted, normalised windows with their targets, and the network and Adam state mid-training."""
    g, rng = _seeds(seed)
    nb = case["nb"]
    win = torch.empty(nb, learned.WIN, dtype=torch.float64, device=DEV).uniform_(0, 1, generator=g).sort(dim=1).values
    win = (win - win[:, :1]) / (win[:, -1:] - win[:, :1])
    pos = torch.empty(nb, 1, dtype=torch.float64, device=DEV).uniform_(0.4, 0.6, generator=g)
    x = torch.cat([win, pos], dim=1).float().contiguous()
    y = torch.empty(nb, dtype=torch.float32, device=DEV).uniform_(0, 1, generator=g)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).to(DEV)  # noqa: E731
    return {"w": dev(learned.init_weights(int(rng.integers(1 << 30)))), "x": x, "y": y,
            "m": dev(rng.standard_normal(learned.MP) * 1e-3), "v": dev(rng.uniform(1e-6, 1e-5, learned.MP)), "step": 100}


def prepare(case, seed):
    e = case["entry"]
    if e == "batch":
        x, off, ks, koff = _batch_inputs(case, seed)
        classes, threads = autotune.load()
        return {"entry": e, "plan": BatchPlan(x, off, ks, koff, classes=classes, block_threads=threads, use_graph=True),
                "nk": int(koff[-1])}
    if e == "train":
        s = _train_inputs(case, seed)
        s.update(entry=e, nb=case["nb"], lib=ggms._lib.load(), g=torch.zeros(learned.MP, device=DEV),
                 loss=torch.zeros(1, device=DEV))
        s["work"] = torch.zeros(int(s["lib"].ggms_mlp_workspace_floats(case["nb"])), device=DEV)
        return s
    x, ks = _select_inputs(case, seed)
    s = {"entry": e, "x": x, "ks": ks, "alg": case["alg"], "nk": case["nk"]}
    s["opts"] = ggms.default_opts(splitter=case["splitter"], schedule=1 if e == "device" else 0)
    if e == "device":
        s["ks"] = torch.from_numpy(ks.view(np.int32)).to(DEV).view(torch.uint32)
        s["out"] = torch.empty(case["nk"], dtype=x.dtype, device=DEV)
    return s


def run(s):
    e = s["entry"]
    if e == "select":
        return ggms.select(s["x"], s["ks"], s["alg"], s["opts"])
    if e == "topk":
        return ggms.topk(s["x"], s["nk"], s["alg"], s["opts"])
    if e == "device":
        return ggms.select_device(s["x"], s["ks"], s["out"], s["alg"], s["opts"])
    if e == "batch":
        s["plan"].launch()
        return s["plan"].out[:s["nk"]]
    lib = s["lib"]
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    ok = lib.ggms_mlp_loss_grad(p(s["w"]), p(s["x"]), p(s["y"]), s["nb"], p(s["g"]), p(s["loss"]), p(s["work"]), None)
    s["step"] += 1
    ok |= lib.ggms_mlp_adam_step(p(s["w"]), p(s["g"]), p(s["m"]), p(s["v"]), s["step"], 2e-3, 0.9, 0.999, 1e-8, None)
    if ok:
        raise RuntimeError("training step failed")
    return {"loss": s["loss"], "grad": s["g"], "w": s["w"], "m": s["m"], "v": s["v"]}


def work(case):
    """Each input read once and each output written once; the network's products for a training step."""
    e = case["entry"]
    if e == "batch":
        # sizes are log-uniform in [2^lo, 2^hi), ranks uniform in 1 .. max_ks: their expected totals
        lo, hi = case["log2_lo"], case["log2_hi"]
        mean = (2.0 ** hi - 2.0 ** lo) / ((hi - lo) * math.log(2))
        b = SIZE[case["dtype"]]
        return {"bytes": case["problems"] * (mean * b + (case["max_ks"] + 1) / 2 * (4 + b)), "flops": 0}
    if e == "train":
        nb, mp = case["nb"], learned.MP
        return {"bytes": 4 * (nb * (learned.MI + 1) + 7 * mp + 1), "flops": 4 * nb * learned.MH * (learned.MI + 1)}
    b = SIZE[case["dtype"]]
    return {"bytes": case["n"] * b + case["nk"] * (4 + b), "flops": 0}


def exact(case, seed):
    e = case["entry"]
    wide = lambda t: t.double() if t.is_floating_point() else t.long()  # noqa: E731
    if e == "batch":
        x, off, ks, koff = _batch_inputs(case, seed)
        kd, got = torch.from_numpy(ks.astype(np.int64)).to(DEV), []
        for i in range(case["problems"]):
            v = x[int(off[i]):int(off[i + 1])]
            v = (v if v.is_floating_point() else v.long()).sort().values
            got.append(wide(v[v.numel() - kd[int(koff[i]):int(koff[i + 1])]]))
        return torch.cat(got)
    if e == "train":
        s = _train_inputs(case, seed)
        w, x, y = s["w"].double(), s["x"].double(), s["y"].double()
        nh, ni = learned.MH, learned.MI
        w1, b1, w2, b2 = w[:nh * ni].view(nh, ni), w[nh * ni:nh * ni + nh], w[nh * ni + nh:nh * ni + 2 * nh], w[-1]
        z = x @ w1.T + b1
        a = z.clamp(min=0)
        p = torch.sigmoid(a @ w2 + b2)
        d = (p - y) * p * (1 - p) / case["nb"]
        dz = torch.where(z > 0, d[:, None] * w2, torch.zeros_like(z))
        g = torch.cat([(dz.T @ x).reshape(-1), dz.sum(0), a.T @ d, d.sum().view(1)])
        f32 = lambda v: float(np.float32(v))  # noqa: E731
        beta1, beta2, t = f32(0.9), f32(0.999), s["step"] + 1
        m = beta1 * s["m"].double() + (1 - beta1) * g
        v = beta2 * s["v"].double() + (1 - beta2) * g * g
        w = w - f32(2e-3) * (m / (1 - beta1 ** t)) / ((v / (1 - beta2 ** t)).sqrt() + f32(1e-8))
        return {"loss": (0.5 * (p - y) ** 2).mean().view(1), "grad": g, "w": w, "m": m, "v": v}
    x, ks = _select_inputs(case, seed)
    v = (x if x.is_floating_point() else x.long()).sort().values
    return wide(v[case["n"] - torch.from_numpy(ks.astype(np.int64)).to(DEV)])
