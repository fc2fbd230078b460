"""Factorisations that prefer one XCD, where they cannot have it: with the wait for it set to nothing every call runs on
the spread workgroups instead, bit-identical; and calls of two streams at once, which compete for the XCDs, end with the
bits that each gives alone."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from spanqr_amd import _lib, borth, kchol, kcholqr_f, kcholqr_f_many, status
from spanqr_amd.plan import Plan, get_plan, stream_handle
from spanqr_amd.qrbench import gen

from checks import assert_bits

pytestmark = pytest.mark.gpu

DEFAULT_TICKS = 1000


@pytest.fixture
def spread():
    _lib.check(_lib.lib().spanqr_debug_place_ticks(0))
    yield
    _lib.check(_lib.lib().spanqr_debug_place_ticks(DEFAULT_TICKS))


# r: the narrowest that prefers one XCD, two owner parts per row and more, the widest; K: the solve as its own launch, in
# the Cholesky's launch with one or two row blocks per workgroup, and one wavefront per row block
@pytest.mark.parametrize("K,r", [(500, 192), (1024, 256), (9000, 256), (768, 512), (4100, 512), (700, 608)])
def test_spread_set_is_bit_exact(cuda, spread, K, r):
    X = gen.ttf_uu(K, r, N=K, seed=r)
    print(f"spread set {K}x{r}", flush=True)
    Q = kcholqr_f(X.to(cuda))
    torch.cuda.synchronize()
    Qo = oracle.orth(X.numpy(), get_plan(K, r, cuda).split_rows)
    assert_bits(Q, Qo, f"{K}x{r}, spread set")
    # the next call on the same plan, one XCD again, and spread once more
    for ticks in (DEFAULT_TICKS, 0):
        _lib.lib().spanqr_debug_place_ticks(ticks)
        assert_bits(kcholqr_f(X.to(cuda)), Qo, f"{K}x{r}, {ticks} ticks on the same plan")


@pytest.mark.parametrize("K,r,n", [(1024, 256, 3), (768, 512, 2), (2048, 512, 12), (800, 544, 8)])
def test_spread_set_of_a_batch(cuda, spread, K, r, n):
    Xs = [gen.ttf_uu(K, r, N=K, seed=i) for i in range(n)]
    print(f"spread set {n} x {K}x{r}", flush=True)
    Qs = kcholqr_f_many([X.to(cuda) for X in Xs])
    torch.cuda.synchronize()
    for i in (0, n - 1):
        assert_bits(Qs[i], oracle.orth(Xs[i].numpy(), get_plan(K, r, cuda).split_rows), f"matrix {i} of the batch")


def test_batch_plan_that_is_spread(cuda):
    """17 matrices of 416 columns take one launch spread and two on XCDs of their own; called with two, the plan's solve
    runs in the Cholesky's launch, whose kernel is the one-XCD one with no set on one XCD"""
    K, r, n = 1000, 416, 2
    Xs = [gen.bench_input(K, r, seed=i).to(cuda) for i in range(n)]
    Qs = [torch.empty_like(X) for X in Xs]
    plan = Plan(K, r, cuda.index, 17)
    assert plan.chol_batch == 17

    def arr(ts):
        return (ctypes.c_void_p * n)(*[t.data_ptr() for t in ts])

    print(f"spread batch plan {n} of 17 x {K}x{r}", flush=True)
    for _ in range(2):
        _lib.check(_lib.lib().spanqr_orth_batched_f32(plan.handle, n, arr(Xs), r, arr(Qs), r, 5e-7, 1e-7, 1e-8, 2,
                                                      stream_handle(cuda)))
        torch.cuda.synchronize()
        for X, Q in zip(Xs, Qs):
            assert_bits(Q, oracle.orth(X.cpu().numpy(), plan.split_rows), "spread batch plan")
    plan.close()


@pytest.mark.parametrize("n", [192, 512, 608])
def test_spread_set_of_the_cholesky_kernels(cuda, spread, n):
    rng = np.random.default_rng(n)
    X = rng.standard_normal((n + 40, n))
    G = X.T @ X
    print(f"spread set chol32, chol64 n={n}", flush=True)
    L, Li = kchol.chol32(torch.from_numpy(G.astype(np.float32)).to(cuda), 1e-6)
    for x, y, what in zip((L, Li), oracle.chol(G.astype(np.float32), np.float32(1e-6)), ("L", "Li")):
        assert_bits(x, y, f"chol32 {what}")
    out = kchol.chol64(torch.from_numpy(G).to(cuda), 1e-12)
    kchol.status(n, cuda)
    for x, y, what in zip(out, oracle.chol64(G, 1e-12), ("L", "Li", "Lf", "Lif")):
        assert np.array_equal(x.cpu().numpy(), y), f"chol64 {what}"


def test_two_streams_at_once(cuda):
    """fp32 calls whose workgroups fill most of an XCD, tall ones whose solve fills the device, blocked ones and fp64
    factorisations, on two streams that are never ordered against each other"""
    shapes = [(768, 512), (17408, 256), (2048, 512), (1024, 256)]
    Xs = [gen.ttf_uu(K, r, N=K, seed=i).to(cuda) for i, (K, r) in enumerate(shapes)]
    W = gen.ttf_uu(3000, 768, N=3000, seed=9).to(cuda)
    A = torch.randn(600, 512, device=cuda, dtype=torch.float64)
    G = A.T.contiguous() @ A
    want = [kcholqr_f(X) for X in Xs] + [borth(W, 256)] + list(kchol.chol64(G, 1e-12))
    streams = [torch.cuda.Stream(cuda), torch.cuda.Stream(cuda)]
    got = [[], []]
    for s in streams:   # the plans (their creation synchronises)
        with torch.cuda.stream(s):
            for X in Xs:
                kcholqr_f(X)
            borth(W, 256)
            kchol.chol64(G, 1e-12)
    torch.cuda.synchronize()
    print("two streams", flush=True)
    for k in range(5):
        for s, out in zip(streams, got):
            with torch.cuda.stream(s):
                out.append([kcholqr_f(X) for X in Xs] + [borth(W, 256)] + list(kchol.chol64(G, 1e-12)))
    torch.cuda.synchronize()
    for i, (s, out) in enumerate(zip(streams, got)):
        for k, qs in enumerate(out):
            for j, (q, w) in enumerate(zip(qs, want)):
                assert torch.equal(q, w), f"stream {i}, round {k}, result {j}"
        with torch.cuda.stream(s):
            status(Xs[-1])
            kchol.status(512, cuda)
