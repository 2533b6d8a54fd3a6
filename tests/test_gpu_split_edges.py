"""The matrix-core f32 convolution and Gemm at the edges of what their split operands hold: what non-finite values touch and what
they cost, pooled tilings, and sums of few terms."""
import time

import numpy as np
import pytest

from oracle import oracle as zo

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import gpu_util
    return gpu_util


def _layer(N, C, H, W, K, kh, kw, seed=0):
    g = np.random.default_rng(N + C + K + seed)
    x = g.standard_normal((N, C, H, W), dtype=np.float32)
    w = (np.abs(g.standard_normal((K, C, kh, kw))) * np.sqrt(2.0 / (C * kh * kw))).astype(np.float32)
    return x, w, (g.standard_normal(K) * 0.1).astype(np.float32)


def _conv(G, x, w, b, pads, act=None):
    args = ([1, 1], pads, [1, 1], 1, "NOTSET")
    y = G.dev(np.full(G.tm.get_convolution_output_shape(x.shape, w.shape, *args[:3], "NOTSET"), 7.0, np.float32))
    G.tm.conv_lean(G.dev(x), G.dev(w), y, G.dev(b), *args, fuse_act=act)
    assert G.tm.context().kernel_name().startswith("conv_f32_split_kernel<"), G.tm.context().kernel_name()
    return G.host(y)


# tiles of one to five 32-position blocks, whole and ragged channel blocks, paired taps and 1x1 filters
@pytest.mark.parametrize("N,C,H,W,K,k", [(2, 24, 16, 16, 40, 3), (256, 32, 28, 28, 64, 3), (200, 32, 14, 14, 200, 3), (3, 20, 31, 22, 50, 5),
                                         (4, 96, 13, 11, 130, 1), (64, 33, 30, 29, 32, 3)])
@pytest.mark.parametrize("act", [None, "relu"])
def test_conv_non_finite_values_leave_the_other_outputs_alone(G, N, C, H, W, K, k, act):
    x, w, b = _layer(N, C, H, W, K, k, k)
    pads = [k // 2] * 4
    clean = _conv(G, x, w, b, pads, act)
    b2 = b.copy()
    b2[3], b2[K - 1] = np.nan, np.inf
    y = _conv(G, x, w, b2, pads, act)
    rest = [c for c in range(K) if c not in (3, K - 1)]
    np.testing.assert_array_equal(y[:, rest], clean[:, rest])
    assert (y[:, 3] == 0).all() if act else np.isnan(y[:, 3]).all()
    assert np.isposinf(y[:, K - 1]).all()
    x2 = x.copy()
    spots = [(0, H // 2, W // 2, np.inf), (N - 1, H - 1, 0, np.nan), (N // 2, 0, W - 1, np.float32(3.4e38))]
    for n, h, v, val in spots:
        x2[n, C - 1, h, v] = val
    y = _conv(G, x2, w, b, pads, act)
    hit = np.zeros((N, H, W), bool)
    for n, h, v, _ in spots:
        hit[n, max(h - k // 2, 0):h + k // 2 + 1, max(v - k // 2, 0):v + k // 2 + 1] = True
    keep = np.broadcast_to(~hit[:, None], y.shape)
    np.testing.assert_array_equal(y[keep], clean[keep])
    for n in sorted({s[0] for s in spots}):
        with np.errstate(all="ignore"):
            ref = zo.Conv(x2[n:n + 1], w, b, [1, 1], pads, [1, 1], 1, "NOTSET")[0]
        np.testing.assert_allclose(y[n], zo.ReLU(ref) if act else ref, rtol=G.RTOL, atol=G.ATOL)


def _time(G, f):
    import torch
    f()
    torch.cuda.synchronize()
    best = 1e9
    for _ in range(5):
        t = time.perf_counter()
        f()
        torch.cuda.synchronize()
        best = min(best, time.perf_counter() - t)
    return best


def test_a_non_finite_value_costs_no_multiple_of_the_layer(G):
    """A NaN bias is an addend like others; one infinite input touches nine positions of one image.  Measured 1.0 and 1.4 times the
    clean layer; each lane by itself term by term took 30 to 250 times."""
    import torch
    x, w = torch.randn(256, 64, 56, 56, device="cuda:0"), torch.randn(64, 64, 3, 3, device="cuda:0") * 0.05
    b, y = torch.randn(64, device="cuda:0"), torch.zeros(256, 64, 56, 56, device="cuda:0")
    call = lambda: G.tm.conv_lean(x, w, y, b, [1, 1], [1] * 4, [1, 1], 1, "NOTSET")
    clean = _time(G, call)
    b[3] = float("nan")
    assert _time(G, call) < 4 * clean
    b[3] = 0.0
    x[5, 0, 20, 20] = float("inf")
    assert _time(G, call) < 8 * clean
    a, m = torch.randn(1, 1, 4096, 1600, device="cuda:0"), torch.randn(1, 1, 1600, 512, device="cuda:0")
    z = torch.zeros(1, 1, 4096, 512, device="cuda:0")
    call = lambda: G.tm.gemm_lean(a, m, None, 1.0, 1.0, False, False, z)
    clean = _time(G, call)
    a[..., 7] = float("nan")  # every row; measured 5 times, each lane by itself 100 times
    assert _time(G, call) < 25 * clean


# ---- fused 2x2/2 max pool: filters of other sizes, strips of wide images, odd sizes -------------------------------------------
POOLED = [
    # N, C, H, W, K, (kh, kw), pads
    (3, 80, 13, 11, 40, (1, 1), [0, 0, 0, 0]),    # 1x1: four channel groups a step, odd sizes
    (2, 12, 15, 14, 33, (5, 5), [2, 2, 2, 2]),    # 25 taps in pairs
    (2, 40, 12, 17, 20, (2, 3), [0, 1, 1, 1]),    # 6 taps of 16 channels
    (1, 33, 9, 1501, 64, (3, 3), [1, 1, 1, 1]),   # a pooled row too wide for LDS: strips, the last one ragged
    (70, 16, 7, 7, 96, (3, 3), [0, 0, 0, 0]),     # several images a tile
]


def _pooled(G, x, w, b, pads, relu):
    N, K = x.shape[0], w.shape[0]
    oh, ow = x.shape[2] + pads[0] + pads[2] - w.shape[2] + 1, x.shape[3] + pads[1] + pads[3] - w.shape[3] + 1
    W_, B_ = G.dev(w), G.dev(b)
    shape = (N, K, oh // 2, ow // 2)
    plan = G.tm.ConvPlan(x.shape, W_, B_, shape, [1, 1], pads, [1, 1], 1, "NOTSET", "relu" if relu else None, True)
    y = G.dev(np.full(shape, np.nan, np.float32))
    plan(G.dev(x), y)
    assert G.tm.context().kernel_name().startswith("conv_f32_split_kernel<"), G.tm.context().kernel_name()
    assert G.tm.context().kernel_name().endswith(",true,true>"), G.tm.context().kernel_name()
    y = G.host(y)
    plan.close()
    return y


def _pooled_ref(x, w, b, pads, relu):
    with np.errstate(all="ignore"):
        c = zo.Conv(x, w, b, [1, 1], pads, [1, 1], 1, "NOTSET")
    return zo.onnx_maxpool(zo.ReLU(c) if relu else c, [2, 2], [2, 2], [1, 1], [0, 0, 0, 0])


@pytest.mark.parametrize("case", POOLED, ids=[str(i) for i in range(len(POOLED))])
@pytest.mark.parametrize("relu", [False, True])
def test_conv_split_pooled_tilings_vs_oracle(G, case, relu):
    N, C, H, W, K, (kh, kw), pads = case
    x, w, b = _layer(N, C, H, W, K, kh, kw)
    np.testing.assert_allclose(_pooled(G, x, w, b, pads, relu), _pooled_ref(x, w, b, pads, relu), rtol=G.RTOL, atol=G.ATOL)


@pytest.mark.parametrize("case", POOLED, ids=[str(i) for i in range(len(POOLED))])
@pytest.mark.parametrize("relu", [False, True])
def test_conv_split_pooled_non_finite_values(G, case, relu):
    N, C, H, W, K, (kh, kw), pads = case
    x, w, b = _layer(N, C, H, W, K, kh, kw, 1)
    clean = _pooled(G, x, w, b, pads, relu)
    x[0, 2, H // 2, W // 2], x[N - 1, C - 1, 1, W - 2], x[0, 0, 0, 0] = np.inf, np.float32(3.4e38), -np.inf
    y, ref = _pooled(G, x, w, b, pads, relu), _pooled_ref(x, w, b, pads, relu)
    assert np.isposinf(ref).any()
    np.testing.assert_allclose(y, ref, rtol=G.RTOL, atol=G.ATOL)
    if N > 2:
        np.testing.assert_array_equal(y[1:N - 1], clean[1:N - 1])
    b[3] = np.nan
    z = _pooled(G, x, w, b, pads, relu)
    others = [c for c in range(K) if c != 3]
    np.testing.assert_array_equal(z[:, others], y[:, others])
    assert (z[:, 3] == 0).all() if relu else np.isnan(z[:, 3]).all()


# ---- Gemm: sums of few terms --------------------------------------------------------------------------------------------------
@pytest.mark.parametrize("M,N", [(70, 66), (1, 17), (200, 33), (64, 128)])
@pytest.mark.parametrize("K", [1, 2, 3, 7, 8, 9, 15, 16, 17])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
def test_gemm_of_few_terms(G, M, N, K, ta, tb):
    """One product is rounded once.  More: never further from 64 bits (2-norm) than the chain of f32 multiply-adds."""
    g = np.random.default_rng(M + N + K)
    a, b = g.standard_normal((M, K)).astype(np.float32), g.standard_normal((K, N)).astype(np.float32)
    a[:, 0] = np.float32(1.0038986)  # 1 + 2^-8 - 2^-17: terms as large as they get, the same sign in every product
    b[0, ::2] = np.float32(1.0038986)
    y = G.dev(np.full((1, 1, M, N), np.nan, np.float32))
    G.tm.gemm_lean(G.dev((a.T if ta else a)[None, None].copy()), G.dev((b.T if tb else b)[None, None].copy()), None, 1.0, 1.0, ta, tb, y)
    assert G.tm.context().kernel_name().startswith("gemm_f32_split_kernel<1,1,%d," % (0 if K <= 16 else 4))
    y = G.host(y)[0, 0]
    if K == 1:
        np.testing.assert_array_equal(y, a * b)
        return
    exact = a.astype(np.float64) @ b.astype(np.float64)
    chain = np.zeros((M, N), np.float32)
    for k in range(K):  # (a product of two f32 is exact in 64 bits; the sum's rounding there is far below f32's)
        chain = (chain.astype(np.float64) + a[:, k:k + 1].astype(np.float64) * b[k].astype(np.float64)).astype(np.float32)
    err, ref = np.linalg.norm(y - exact), np.linalg.norm(chain - exact)
    assert err <= 1.02 * ref, (err / ref)


def test_gemm_of_few_terms_non_finite_and_unaligned(G):
    import torch
    g = np.random.default_rng(5)
    a, b = g.standard_normal((1, 1, 37, 16), dtype=np.float32), np.abs(g.standard_normal((1, 1, 16, 70), dtype=np.float32))
    a[0, 0, 3, 2], a[0, 0, 20, 15], a[0, 0, 36, 0] = np.inf, np.nan, np.float32(3e38)
    flat = torch.zeros(a.size + 4, device="cuda:0")
    A = flat[1:1 + a.size].view(a.shape)
    A.copy_(torch.from_numpy(a))
    y = G.dev(np.full((1, 1, 37, 70), 7.0, np.float32))
    G.tm.gemm_lean(A, G.dev(b), None, 1.0, 1.0, False, False, y)
    with np.errstate(all="ignore"):
        np.testing.assert_allclose(G.host(y), zo.gemm(a, b, None, 1.0, 1.0, False, False), rtol=G.RTOL, atol=G.ATOL)


# ---- operands whose left-out term products are as large as they get ------------------------------------------------------------
def test_split_error_bound_of_equal_operands(G):
    """1.0038986 splits into 1 + 2^-8 - 2^-17: 2^-24 of every product is left out, always with the same sign.  The result may be
    that far off, plus f32 roundings of n products of one sign: one per 16, each at most half a unit of the sum so far."""
    v = np.float32(1.0038986)
    for C, k in [(20, 3), (12, 3), (64, 1)]:
        n = C * k * k
        x, w = np.full((2, C, 9, 9), v, np.float32), np.full((33, C, k, k), v, np.float32)
        y = G.host(G.tm.Conv(G.dev(x), G.dev(w), None, [1, 1], [0, 0, 0, 0], [1, 1], 1, "NOTSET"))
        assert G.tm.context().kernel_name().startswith("conv_f32_split_kernel<")
        exact = n * np.float64(v) ** 2
        assert np.abs(y - exact).max() <= exact * 2.0 ** -24 * (1.05 + 6 * -(-n // 16) / 2)
    a, b = np.full((1, 1, 70, 1600), v, np.float32), np.full((1, 1, 1600, 66), v, np.float32)
    y = G.dev(np.zeros((1, 1, 70, 66), np.float32))
    G.tm.gemm_lean(G.dev(a), G.dev(b), None, 1.0, 1.0, False, False, y)
    exact = 1600 * np.float64(v) ** 2
    assert np.abs(G.host(y) - exact).max() <= exact * 2.0 ** -24 * (1.05 + 6 * 100 / 2)


# ---- rows of 2^22 elements and more: the kernel with 64-bit addresses, in every storage order -----------------------------------
@pytest.mark.parametrize("M,K,N,ta,tb", [(3, 5, (1 << 22) + 3, False, False), ((1 << 22) + 5, 3, 17, True, False),
                                         ((1 << 22) + 1, 3, 18, True, True), (5, (1 << 22) + 2, 19, False, True)])
def test_gemm_long_rows_in_every_storage_order(G, M, K, N, ta, tb):
    import torch
    t = torch.Generator(device="cuda:0").manual_seed(M + N)
    a = torch.randn((K, M) if ta else (M, K), generator=t, device="cuda:0")
    b = torch.randn((N, K) if tb else (K, N), generator=t, device="cuda:0")
    y = torch.full((1, 1, M, N), float("nan"), device="cuda:0")
    G.tm.gemm_lean(a[None, None], b[None, None], None, 1.0, 1.0, ta, tb, y)
    flags = "%s,%s>" % ("false" if ta else "true", "true" if tb else "false")
    assert G.tm.context().kernel_name().startswith("gemm_f32_mfma_kernel<") and G.tm.context().kernel_name().endswith(flags)
    ref = (a.T if ta else a).double().cpu().numpy() @ (b.T if tb else b).double().cpu().numpy()
    rms = np.sqrt(np.mean(ref ** 2))
    assert np.sqrt(np.mean((G.host(y)[0, 0] - ref) ** 2)) < np.sqrt(K) * 2.0 ** -24 * rms


@pytest.mark.parametrize("M,K,N,tile", [(4001, 1601, 509, "<2,1,"), (6001, 997, 515, "<2,2,")])
@pytest.mark.parametrize("ta,tb", [(False, False), (True, True)])
def test_gemm_large_tiles_non_finite_values(G, M, K, N, tile, ta, tb):
    """Blocks computed again at ragged edges of the larger tiles: the values 64 bits give, non-finite ones among them."""
    g = np.random.default_rng(M)
    a, b = g.standard_normal((M, K), dtype=np.float32), (np.abs(g.standard_normal((K, N))) * 0.01).astype(np.float32)
    a[M - 1, 3], a[17, 5], a[M - 2, 0], b[7, N - 1] = np.inf, np.nan, np.float32(3e38), -np.inf
    y = G.dev(np.full((1, 1, M, N), 7.0, np.float32))
    G.tm.gemm_lean(G.dev((a.T if ta else a)[None, None].copy()), G.dev((b.T if tb else b)[None, None].copy()), None, 1.0, 1.0, ta, tb, y)
    assert tile in G.tm.context().kernel_name()
    with np.errstate(all="ignore"):
        ref = a.astype(np.float64) @ b.astype(np.float64)
    np.testing.assert_allclose(G.host(y)[0, 0], ref, rtol=G.RTOL, atol=G.ATOL)
