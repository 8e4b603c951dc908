"""The work a user of this package has it do, as cases that can be timed and
compared: Ozaki products, Gram matrices, residuals and solves through the
public entry points, at the sizes of the tests and the benchmark suite and
over the ranges around them.

  listed()           the fixed cases
  draw(rng)          one more case of the same ranges
  prepare(case, s)   the inputs a program has in hand before the call
  run(state)         one call
  work(case)         bytes and operations the path cannot do without
  tolerance(case)    how far another correct implementation may be
  exact(case, s)     the same result in plain 64-bit arithmetic
"""

import math

import numpy as np
import torch

import ozaki_jax_amd as ozk

_PRESETS = {"high": (4, 1), "medium": (3, 1), "max": (5, 4)}

# Work of the largest listed case: the 8192^3 product with 24 slice pairs.
_MOST_FLOPS = 24 * 2.0 * 8192 ** 3
_MOST_ELEMENTS = 64 * 1024 * 1024 + 1


def listed():
    return [
        # The smallest products, where launches and latency count: 256^3 on
        # tensors already on the GPU ...
        {"name": "matmul_256", "op": "matmul", "n": 256, "k": 256, "m": 256,
         "precision": "high", "accumulation": "fused", "data": "normal"},
        # ... and the package's default call, NumPy arrays through the host
        # pipeline (FP64 extraction, eight slices), transfers included.
        {"name": "host_256", "op": "host", "n": 256, "k": 256, "m": 256, "slices": 8,
         "entry": "matmul_numpy", "data": "normal"},
        # An ordinary product of odd sizes.
        {"name": "matmul_1000x1531x777", "op": "matmul", "n": 1000, "k": 1531, "m": 777,
         "precision": "high", "accumulation": "fused", "data": "normal"},
        # The host pipeline on GPU tensors at a size where its kernels count.
        {"name": "host_2048x1024x2048", "op": "host", "n": 2048, "k": 1024, "m": 2048,
         "slices": 8, "entry": "matmul", "data": "normal"},
        # Square products on BF16 planes (K <= 4096) and, the headline
        # benchmark, on INT8 planes.
        {"name": "matmul_4096", "op": "matmul", "n": 4096, "k": 4096, "m": 4096,
         "precision": "high", "accumulation": "fused", "data": "normal"},
        {"name": "matmul_8192", "op": "matmul", "n": 8192, "k": 8192, "m": 8192,
         "precision": "high", "accumulation": "fused", "data": "normal"},
        # The other presets, on entries of a wide range: medium in the FP64
        # block order at ragged sizes, max in its three sweeps.
        {"name": "matmul_medium_3001x6000x2500", "op": "matmul", "n": 3001, "k": 6000,
         "m": 2500, "precision": "medium", "accumulation": "host", "data": "wide"},
        {"name": "matmul_max_2048x8192x2048", "op": "matmul", "n": 2048, "k": 8192,
         "m": 2048, "precision": "max", "accumulation": "fused", "data": "wide"},
        # A long contraction: few output tiles, extraction-heavy.
        {"name": "matmul_1024x65536x1024", "op": "matmul", "n": 1024, "k": 65536, "m": 1024,
         "precision": "high", "accumulation": "fused", "data": "wide"},
        # The Gram matrix and the residual of a tall system.
        {"name": "gram_32768x2048", "op": "gram", "n": 32768, "k": 2048, "precision": "high",
         "data": "normal"},
        {"name": "residual_32768x2048", "op": "residual", "n": 32768, "k": 2048, "m": 1,
         "precision": "high", "data": "normal"},
        # A linear system of condition 1e6: FP32 factorisation and three
        # refinement steps on Ozaki residuals.
        {"name": "solve_4096", "op": "solve", "n": 4096, "m": 1, "precision": "high",
         "cond": 1e6},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """A size spread over the logarithm of its range; half of them as users
    have them (a multiple of 64 where that is inside), half any number."""
    v = _log_int(rng, lo, hi)
    if rng.random() < 0.5 and v >= 128:
        v = v // 64 * 64
    return max(lo, min(hi, v))


def draw(rng):
    op = rng.choice(["matmul"] * 5 + ["host"] * 2 + ["gram", "residual", "solve"])
    data = rng.choice(["normal", "wide"])
    if op == "matmul":
        precision = rng.choice(["high", "high", "high", "medium", "max", "3,2", "4,2"])
        accumulation = rng.choice(["fused", "fused", "host"])
        while True:
            c = {"op": op, "n": _size(rng, 64, 8192), "k": _size(rng, 64, 65536),
                 "m": _size(rng, 64, 8192), "precision": precision,
                 "accumulation": accumulation, "data": data}
            if (work(c)["flops"] <= _MOST_FLOPS and c["n"] * c["k"] <= _MOST_ELEMENTS
                    and c["m"] * c["k"] <= _MOST_ELEMENTS):
                return c
    if op == "host":
        # 8 slices of 7 bits hold an FP64 value up to K = 1024, 9 of 6 above
        k = _size(rng, 64, 4096)
        return {"op": op, "n": _size(rng, 64, 4096), "k": k, "m": _size(rng, 64, 4096),
                "slices": 8 if k <= 1024 else 9, "data": data,
                "entry": rng.choice(["matmul", "matmul_numpy"])}
    precision = rng.choice(["high", "high", "medium", "max"])
    if op == "gram":
        while True:
            c = {"op": op, "n": _size(rng, 64, 65536), "k": _size(rng, 64, 8192),
                 "precision": precision, "data": data}
            if work(c)["flops"] <= _MOST_FLOPS and c["n"] * c["k"] <= _MOST_ELEMENTS:
                return c
    if op == "residual":
        while True:
            c = {"op": op, "n": _size(rng, 64, 65536), "k": _size(rng, 64, 16384),
                 "m": rng.choice([1, 1, 2, 4]), "precision": precision, "data": data}
            if c["n"] * c["k"] <= _MOST_ELEMENTS:
                return c
    return {"op": op, "n": _size(rng, 64, 4096), "m": rng.choice([1, 1, 2, 4]),
            "precision": precision, "cond": rng.choice([1e2, 1e4, 1e6])}


def _entries(gen, shape, data):
    """N(0, 1) entries, or (U - 0.5) exp(2 N): magnitudes over a wide range."""
    kw = {"dtype": torch.float64, "device": "cuda", "generator": gen}
    if data == "normal":
        return torch.randn(shape, **kw)
    u = torch.rand(shape, **kw)
    return (u - 0.5) * torch.exp(2.0 * torch.randn(shape, **kw))


def _precision(case):
    p = case["precision"]
    return tuple(int(v) for v in p.split(",")) if "," in p else p


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    op, n = case["op"], case["n"]
    st = {"case": case}
    if op in ("matmul", "host"):
        st["A"] = _entries(gen, (n, case["k"]), case["data"])
        st["B"] = _entries(gen, (case["k"], case["m"]), case["data"])
        if case.get("entry") == "matmul_numpy":
            st["A"], st["B"] = st["A"].cpu().numpy(), st["B"].cpu().numpy()
    elif op == "gram":
        st["A"] = _entries(gen, (n, case["k"]), case["data"])
    elif op == "residual":
        vec = case["m"] == 1
        st["A"] = _entries(gen, (n, case["k"]), case["data"])
        st["x"] = _entries(gen, (case["k"],) if vec else (case["k"], case["m"]), "normal")
        st["b"] = _entries(gen, (n,) if vec else (n, case["m"]), "normal")
    else:
        # A = Q1 diag(1 .. cond, log-spaced) Q2^T
        q1, _ = torch.linalg.qr(_entries(gen, (n, n), "normal"))
        q2, _ = torch.linalg.qr(_entries(gen, (n, n), "normal"))
        d = torch.logspace(0, math.log10(case["cond"]), n, dtype=torch.float64, device="cuda")
        st["A"] = (q1 * d) @ q2.T.contiguous()
        st["b"] = _entries(gen, (n,) if case["m"] == 1 else (n, case["m"]), "normal")
    return st


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "matmul":
        return ozk.matmul(state["A"], state["B"], pipeline="ondevice",
                          accumulation=case["accumulation"], precision=_precision(case))
    if op == "host":
        entry = ozk.matmul_numpy if case["entry"] == "matmul_numpy" else ozk.matmul
        return entry(state["A"], state["B"], n_slices=case["slices"])
    if op == "gram":
        return ozk.gram(state["A"], precision=_precision(case), mode="ozaki")
    if op == "residual":
        return ozk.residual(state["A"], state["x"], state["b"], precision=_precision(case),
                            mode="ozaki")
    return ozk.solve(state["A"], state["b"], precision=_precision(case),
                     residual_mode="ozaki")


def _pairs(case):
    if case["op"] == "host":
        return case["slices"] * (case["slices"] + 1) // 2
    hi, lo = _PRESETS.get(case["precision"]) or _precision(case)
    return hi * hi + 2 * hi * lo


def work(case):
    op, n = case["op"], case["n"]
    if op in ("matmul", "host"):
        k, m = case["k"], case["m"]
        return {"bytes": 8.0 * (n * k + k * m + n * m), "flops": 2.0 * _pairs(case) * n * k * m}
    if op == "gram":  # symmetric: the products on and above the diagonal
        k = case["k"]
        return {"bytes": 8.0 * (n * k + k * k), "flops": 1.0 * _pairs(case) * n * k * (k + 1)}
    if op == "residual":
        k, m = case["k"], case["m"]
        return {"bytes": 8.0 * (n * k + k * m + 2 * n * m),
                "flops": 2.0 * _pairs(case) * n * k * m}
    # solve: factorisation, four triangular solves, three residuals, each of
    # which reads A or its factor
    m = case["m"]
    return {"bytes": 8.0 * n * n + 4.0 * n * n + 16.0 * n * m,
            "flops": 2.0 / 3.0 * n ** 3 + 4 * 2.0 * n * n * m + 3 * 2.0 * _pairs(case) * n * n * m}


def tolerance(case):
    # Products, Gram matrices and residuals are defined bit by bit: the
    # slices, the exact products of slice pairs and the order in which they
    # are folded.
    if case["op"] != "solve":
        return "exact"
    # Three refinement steps shrink what the FP32 factorisation's rounding
    # left by about cond * 2^-24 * a few each, down to the residual's own
    # error (about 1e-10 of it, 1e-7 for medium).  Stated: four times the
    # difference between this factorisation and another correct one.
    rel = {1e2: 1e-8, 1e4: 2e-7, 1e6: 2.5e-4}[case["cond"]]
    return {"rel": rel + (2e-6 if case["precision"] == "medium" else 0.0)}


def exact(case, seed):
    st = prepare(case, seed)
    op = case["op"]
    if op in ("matmul", "host"):
        if op == "host" or case.get("entry") == "matmul_numpy":
            a, b = (torch.as_tensor(st[v]).cuda() for v in "AB")
            return torch.matmul(a, b).cpu().numpy()
        return torch.matmul(st["A"], st["B"])
    if op == "gram":
        g = torch.matmul(st["A"].T.contiguous(), st["A"])
        return (g + g.T) * 0.5
    if op == "residual":
        return st["b"] - torch.matmul(st["A"], st["x"])
    x = np.linalg.solve(st["A"].cpu().numpy(), st["b"].cpu().numpy())
    return torch.from_numpy(x).cuda()
