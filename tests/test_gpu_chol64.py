"""The fp64 clamped Cholesky (kchol.chol64 -> chol_f64) through the C ABI: L, Li and their fp32 copies bit-identical
to the oracle's fp64 restatement at n = 32..1024 on SPD, rank-deficient, zero and NaN-pivot inputs, tau as a float or
a device tensor, repeat determinism, and no wait that gave up."""
import numpy as np
import pytest
import torch

import oracle
from spanqr_amd import kchol

pytestmark = pytest.mark.gpu


def _bits(a, b, what):
    """bit-identical, except that a NaN matches any NaN: the default NaN differs between the host (sign set) and the
    GPU (canonical positive), and a clamped NaN pivot with a tiny tau overflows into NaNs further down"""
    a = a.detach().cpu().numpy() if isinstance(a, torch.Tensor) else a
    u = np.uint64 if a.dtype == np.float64 else np.uint32
    both_nan = np.isnan(a) & np.isnan(b)
    diff = (np.ascontiguousarray(a).view(u) != np.ascontiguousarray(b).view(u)) & ~both_nan
    assert not diff.any(), f"{what}: {int(diff.sum())} elements differ"


def _case(n, kind, rng):
    if kind == "spd":
        X = rng.standard_normal((n + 50, n)) * np.exp(rng.uniform(-4, 4, n))
        return X.T @ X, 1e-14
    if kind == "rank":
        B = rng.standard_normal((n, n // 4))
        return B @ B.T, 1e-9
    if kind == "zero":
        return np.zeros((n, n)), 1e-30
    X = rng.standard_normal((n + 10, n))
    G = X.T @ X
    G[n // 3, n // 3] = np.nan
    return G, 1e-6


@pytest.mark.parametrize("n,kind", [(32, "spd"), (64, "spd"), (128, "rank"), (256, "spd"), (256, "nan"),
                                    (512, "spd"), (512, "zero"), (1024, "spd")])
def test_chol64_bit_exact(cuda, n, kind):
    rng = np.random.default_rng(n + len(kind))
    G, tau = _case(n, kind, rng)
    print(f"chol64 n={n} {kind}", flush=True)
    L, Li, Lf, Lif = kchol.chol64(torch.from_numpy(G).to(cuda), tau)
    kchol.status(n, cuda)
    Lo, Lio, Lfo, Lifo = oracle.chol64(G, tau)
    _bits(L, Lo, "L")
    _bits(Li, Lio, "Li")
    _bits(Lf, Lfo, "Lf")
    _bits(Lif, Lifo, "Lif")


def test_chol64_tau_tensor_and_repeat(cuda):
    rng = np.random.default_rng(3)
    X = rng.standard_normal((300, 256))
    G = torch.from_numpy(X.T @ X).to(cuda)
    t = torch.tensor([1e-12], device=cuda, dtype=torch.float64)
    a = kchol.chol64(G, t)
    b = kchol.chol64(G, 1e-12)
    c = kchol.chol64(G, t)
    torch.cuda.synchronize()
    for x, y, z in zip(a, b, c):
        assert torch.equal(x, y) and torch.equal(x, z)
    L = a[0].cpu().numpy()
    assert np.abs(L @ L.T - X.T @ X).max() <= 1e-12 * np.abs(X.T @ X).max()


def test_chol64_rejects_bad_inputs(cuda):
    with pytest.raises(TypeError):
        kchol.chol64(torch.zeros(64, 64, device=cuda), 1e-9)          # fp32
    with pytest.raises(ValueError):
        kchol.chol64(torch.zeros(48, 48, device=cuda, dtype=torch.float64), 1e-9)
    with pytest.raises(ValueError):
        kchol.chol64(torch.zeros(1056, 1056, device=cuda, dtype=torch.float64), 1e-9)


@pytest.mark.parametrize("n", [96, 192, 224, 544, 576, 608, 640, 992])
def test_chol64_row_parts(cuda, n):
    """the sizes where the split changes: the first tile row with a workgroup of its own (96), rows of one and of two
    parts (192, 224), a whole XCD in the narrow parts (544), the wider parts that still fit on one (576, 608), the
    workgroups spread over the device (640, 992), with an ill-scaled G and with a pivot row that vanishes in the last tile"""
    rng = np.random.default_rng(n)
    X = rng.standard_normal((n + 9, n)) * np.exp(rng.uniform(-6, 6, n))
    X[:, n - 2] = X[:, 1]
    G = X.T @ X
    out = kchol.chol64(torch.from_numpy(G).to(cuda), 1e-10)
    kchol.status(n, cuda)
    for x, y, what in zip(out, oracle.chol64(G, 1e-10), ("L", "Li", "Lf", "Lif")):
        _bits(x, y, what)


def test_chol64_first_call_captured(cuda):
    """a plan whose first call is captured clears its flags in the graph; eager calls and replays may then alternate"""
    n = 288
    rng = np.random.default_rng(1)
    X = rng.standard_normal((n + 9, n))
    G, t = torch.from_numpy(X.T @ X).to(cuda), torch.tensor([1e-12], device=cuda, dtype=torch.float64)
    want = oracle.chol64(X.T @ X, 1e-12)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        kchol._plan(n, G.device)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            out = kchol.chol64(G, t)
        for k in range(4):
            for o in out:
                o.fill_(float("nan"))
            g.replay()
            eager = kchol.chol64(G, t)
            torch.cuda.synchronize()
            for x, e, y, what in zip(out, eager, want, ("L", "Li", "Lf", "Lif")):
                _bits(x, y, f"{what}, replay {k}")
                _bits(e, y, f"{what}, eager call after replay {k}")
