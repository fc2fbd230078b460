"""The work that programs give this library, as cases that can be timed and compared.

An optimizer of TTF layers calls orth(X) on every layer of every step: X [K, r] is a tall fp32 matrix on the GPU and
the call returns an orthonormal basis of its columns. So most cases are one such call, at the layer sizes of the
models that qrbench names (SHAPES in spanqr_amd/qrbench/gen.py), from the smallest size that is still worth a GPU call
to the 27B layers; then ragged sizes, the full-width and the column-blocked form of the wide layers, a whole step of
24 layers in one call (orth_many), and the two Cholesky kernels that kchol exports, one in fp32 and one in fp64.

A case is {"kind", ...}:
  orth       K, r             orth(X), whatever branch it takes
  kcholqr_f  K, r             kcholf at full width, also where orth would block the columns
  borth      K, r, b, reorth  block Gram-Schmidt with the caller's block width, with or without the second round
  orth_many  K, r, n, K2, r2, n2   two groups of same-shape layers of one step
  chol32, chol64   n          the clamped Cholesky with the inverses of its diagonal tiles
"""
import math

import numpy as np
import torch

from spanqr_amd import borth, kcholqr_f, orth, orth_many
from spanqr_amd.kchol import chol32, chol64

EPS = 5e-7        # the dust that kcholqr_f adds by default, relative to the scaled X
DUST_SEED = 20261018
CHOL_TAU = 1e-12  # pivot floor of the Cholesky cases: below every pivot of a well-conditioned G


def listed():
    return [
        # the smallest call: nothing but launches and latency
        {"name": "orth_256x128", "kind": "orth", "K": 256, "r": 128},
        # attention layer of the 0.8B model
        {"name": "orth_1024x256", "kind": "orth", "K": 1024, "r": 256},
        # attention and down_proj layers of the 110M model
        {"name": "orth_768x512", "kind": "orth", "K": 768, "r": 512},
        {"name": "orth_2048x512", "kind": "orth", "K": 2048, "r": 512},
        # down_proj layer of the 27B model: the tallest X
        {"name": "orth_17408x256", "kind": "orth", "K": 17408, "r": 256},
        # odd row count, r an odd multiple of 32: the last tile of everything is ragged
        {"name": "orth_3001x736", "kind": "orth", "K": 3001, "r": 736},
        # the widest full-width kcholf
        {"name": "kcholqr_f_2048x1024", "kind": "kcholqr_f", "K": 2048, "r": 1024},
        # 27B layers kept at a wider rank: block Gram-Schmidt over 256-column blocks
        {"name": "orth_5120x1024", "kind": "orth", "K": 5120, "r": 1024},
        {"name": "orth_17408x2048", "kind": "orth", "K": 17408, "r": 2048},
        # one optimizer step of the 110M model: all 24 layers in one call
        {"name": "step_24_layers", "kind": "orth_many", "K": 768, "r": 512, "n": 12, "K2": 2048, "r2": 512, "n2": 12},
        # the Cholesky kernels on their own
        {"name": "chol32_512", "kind": "chol32", "n": 512},
        {"name": "chol64_512", "kind": "chol64", "n": 512},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: every kind over its whole range. K is any integer from 1.25 r up (a square random X has no
    bounded condition number) and no case does more than the largest listed one."""
    kind = rng.choice(["orth", "orth", "orth", "orth", "orth", "full", "wide", "wide", "borth", "orth_many", "chol32",
                       "chol64"])
    if kind == "orth":                       # kcholf below and at 512 columns
        r = 32 * _log_int(rng, 1, 16)
        return {"kind": "orth", "K": _log_int(rng, r * 5 // 4, 20000), "r": r}
    if kind == "full":                       # kcholf at full width above 512 columns
        r = 32 * rng.randint(17, 32)
        return {"kind": "kcholqr_f", "K": _log_int(rng, r * 5 // 4, 8192), "r": r}
    if kind == "wide":                       # orth over 256-column blocks
        r = 256 * rng.randint(3, 8)
        return {"kind": "orth", "K": _log_int(rng, r * 5 // 4, 17408), "r": r}
    if kind == "borth":
        b = 32 * _log_int(rng, 4, 16)
        r = b * rng.randint(2, 1024 // b)
        return {"kind": "borth", "K": _log_int(rng, r * 5 // 4, 12000), "r": r, "b": b, "reorth": rng.random() < 0.5}
    if kind == "orth_many":
        r, r2 = 32 * _log_int(rng, 4, 16), 32 * _log_int(rng, 4, 16)
        return {"kind": "orth_many", "K": _log_int(rng, r * 5 // 4, 4096), "r": r, "n": rng.randint(2, 16),
                "K2": _log_int(rng, r2 * 5 // 4, 4096), "r2": r2, "n2": rng.randint(1, 16)}
    return {"kind": kind, "n": 32 * _log_int(rng, 1, 32)}


def _layers(case):
    if case["kind"] == "orth_many":
        return [(case["K"], case["r"])] * case["n"] + [(case["K2"], case["r2"])] * case["n2"]
    return [(case["K"], case["r"])]


def _matrix(K, r, g, dtype=torch.float32):
    """[K, r]: Gaussian rows, column scales log-spaced over two decades (the spread of a TTF update's singular values
    that a 32-bit result still resolves), mixed by a reflection so that every column holds every scale."""
    X = torch.randn(K, r, generator=g, device="cuda", dtype=dtype)
    X *= torch.logspace(0, -2, r, device="cuda", dtype=dtype)[torch.randperm(r, generator=g, device="cuda")]
    v = torch.randn(r, 1, generator=g, device="cuda", dtype=dtype)
    v /= v.norm()
    return (X - 2.0 * (X @ v) @ v.T).contiguous()


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    if case["kind"] in ("chol32", "chol64"):
        n = case["n"]
        A = torch.randn(2 * n, n, generator=g, device="cuda", dtype=torch.float64)
        A *= torch.logspace(0, -1, n, device="cuda", dtype=torch.float64)[torch.randperm(n, generator=g, device="cuda")]
        G = A.T.contiguous() @ A / (2 * n)
        return {"case": case, "G": G.float() if case["kind"] == "chol32" else G}
    return {"case": case, "X": [_matrix(K, r, g) for K, r in _layers(case)]}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "orth":
        return orth(state["X"][0])
    if kind == "kcholqr_f":
        return kcholqr_f(state["X"][0])
    if kind == "borth":
        return borth(state["X"][0], case["b"], case["reorth"])
    if kind == "orth_many":
        return orth_many(state["X"])
    return (chol32 if kind == "chol32" else chol64)(state["G"], CHOL_TAU)


def _blocks(case):
    """the block width where the columns are blocked (orth: above 512 columns, multiples of 256), else None"""
    K, r = _layers(case)[0]
    if case["kind"] == "borth":
        return case["b"]
    return 256 if case["kind"] == "orth" and r > 512 and r % 256 == 0 else None


def _kcholf_flops(K, r):
    # three passes of Gram and solve, two polish Grams and products, three factorisations
    return 8 * K * r * (r + 1) + 4 * K * r * r + r ** 3


def work(case):
    if case["kind"] in ("chol32", "chol64"):
        n, w = case["n"], 4 if case["kind"] == "chol32" else 8
        out = w * (n * n + 32 * n)
        return {"bytes": w * n * n // 2 + out + (out // 2 if w == 8 else 0), "flops": n ** 3 // 3 + n * 32 * 32 // 3}
    nbytes = sum(8 * K * r for K, r in _layers(case))
    b = _blocks(case)
    if b is None:
        return {"bytes": nbytes, "flops": sum(_kcholf_flops(K, r) for K, r in _layers(case))}
    (K, r), = _layers(case)
    second = case.get("reorth", True)
    flops = r // b * _kcholf_flops(K, b)
    for j in range(b, r, b):
        flops += (3 if second else 2) * 4 * K * j * b + (_kcholf_flops(K, b) if second else 0)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # About four times the largest error against exact() over 1500 draws: 1.02e-6 for a Q, 4.5e-7 for an fp32 factor;
    # 8e-16 for an fp64 factor, but its fp32 copies may differ in the last bit of a value next to a tie (1.7e-11 seen).
    return {"rel": {"chol32": 1.5e-6, "chol64": 1e-9}.get(case["kind"], 4e-6)}


# ---- the same results in 64 bits ----

def _dust(K, r):
    """The dust matrix: element n = k r + c is the sum of the twelve 32-bit halves of six splitmix64 outputs, centred,
    scaled to unit variance and rounded to fp32; then unit columns, rounded to fp32."""
    def mix(z):
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        return z ^ (z >> np.uint64(31))

    with np.errstate(over="ignore"):
        key = mix(np.array([DUST_SEED], dtype=np.uint64))
        Z = np.empty((K, r), dtype=np.float64)
        step = max(1, (1 << 20) // r)
        for k0 in range(0, K, step):
            n = np.arange(k0 * r, min(K, k0 + step) * r, dtype=np.uint64)
            s = np.zeros(n.shape, dtype=np.int64)
            for j in range(1, 7):
                w = mix(key + (np.uint64(6) * n + np.uint64(j)) * np.uint64(0x9E3779B97F4A7C15))
                s += (w & np.uint64(0xFFFFFFFF)).astype(np.int64) + (w >> np.uint64(32)).astype(np.int64)
            z = ((s - 6 * 4294967295).astype(np.float64) * 2.0 ** -32).astype(np.float32)
            Z[k0:k0 + step] = z.reshape(-1, r)
    Z /= np.sqrt((Z * Z).sum(axis=0))
    return torch.from_numpy(Z.astype(np.float32).astype(np.float64))


def _scale(X):
    m = float(X.abs().max())
    return 2.0 ** -round(math.log2(m)) if m > 0 else 1.0


def _kcholf(X, Z):
    """the Q factor with a positive diagonal of s X + eps Z, to which the shifted passes and the polish converge"""
    Q, R = torch.linalg.qr(_scale(X) * X + EPS * Z)
    d = torch.sign(torch.diagonal(R))
    return Q * torch.where(d == 0, torch.ones_like(d), d)


def _borth(X, b, second):
    K, r = X.shape
    Z, s = _dust(K, r), _scale(X)
    Q = torch.empty_like(X)
    for j in range(0, r, b):
        P, Zj = Q[:, :j], Z[:, j:j + b]
        W = s * X[:, j:j + b]
        for _ in range(2 if j else 0):
            W = W - P @ (P.T @ W)
        W = _kcholf(W, Zj)
        if j and second:
            W = _kcholf(W - P @ (P.T @ W), Zj)
        Q[:, j:j + b] = W
    return Q


def exact(case, seed):
    state = prepare(case, seed)
    if case["kind"] in ("chol32", "chol64"):
        n = case["n"]
        L = torch.linalg.cholesky(state["G"].double().cpu())
        t = [torch.linalg.inv(L[i:i + 32, i:i + 32]) for i in range(0, n, 32)]
        Li = torch.cat([torch.tril(x) for x in t])
        return (L, Li) if case["kind"] == "chol32" else (L, Li, L.float(), Li.float())
    X = [x.double().cpu() for x in state["X"]]
    b = _blocks(case)
    if b is not None:
        return _borth(X[0], b, case.get("reorth", True))
    dust = {s: _dust(*s) for s in set(_layers(case))}
    Q = [_kcholf(x, dust[tuple(x.shape)]) for x in X]
    return Q if case["kind"] == "orth_many" else Q[0]
