"""f32 Gemms whose K is cut among workgroups: parts of one step, parts of uneven length, blocks that lie outside the matrix, sums that
come out non-finite, and the same bits whichever workgroup finishes a block."""
import numpy as np
import pytest
import torch

from oracle import oracle as zo

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import gpu_util
    return gpu_util


def _inputs(M, K, N):
    g = np.random.default_rng(M + K + N)
    return g.standard_normal((1, 1, M, K), dtype=np.float32), (g.standard_normal((1, 1, K, N)) * np.sqrt(2.0 / K)).astype(np.float32)


# K of a few steps, just past a whole number of them, one that no number of parts divides, and the longest cut into the most parts
SHAPES = [(1, 200, 24), (33, 225, 65), (64, 256, 17), (65, 1601, 129), (7, 4096, 40), (130, 997, 333), (333, 1600, 512), (1, 9001, 1000)]


@pytest.mark.parametrize("ta", [False, True])
@pytest.mark.parametrize("tb", [False, True])
@pytest.mark.parametrize("M,K,N", SHAPES)
def test_gemm_cut_k_vs_64_bits(G, M, K, N, ta, tb):
    a, b = _inputs(M, K, N)
    c = np.random.default_rng(1).standard_normal((1, 1, M, N)).astype(np.float32)
    A, B = G.dev(np.swapaxes(a, -1, -2).copy() if ta else a), G.dev(np.swapaxes(b, -1, -2).copy() if tb else b)
    runs = []
    for _ in range(3):
        y = G.dev(np.full((1, 1, M, N), np.nan, np.float32))
        G.tm.gemm_lean(A, B, G.dev(c), 1.5, 0.5, ta, tb, y, "relu")
        runs.append(G.host(y)[0, 0])
    np.testing.assert_array_equal(runs[0], runs[1])
    np.testing.assert_array_equal(runs[0], runs[2])
    full = 1.5 * (a[0, 0].astype(np.float64) @ b[0, 0].astype(np.float64)) + 0.5 * c[0, 0]
    # a random walk of K f32 roundings; a part that is missing or counted twice would show at the size of the result
    rms = np.sqrt(np.mean(full ** 2))
    d = runs[0] - np.maximum(full, 0)
    assert np.sqrt(np.mean(d ** 2)) < np.sqrt(K) * 2.0 ** -24 * rms
    assert np.abs(d).max() < 8 * np.sqrt(K) * 2.0 ** -24 * rms


def test_gemm_cut_k_non_finite(G):
    a, b = _inputs(70, 1000, 68)
    b = np.abs(b)
    a[0, 0, 3, 5], a[0, 0, 9, 999], a[0, 0, 20, 400], a[0, 0, 69, 600] = np.inf, np.nan, np.float32(3.0e38), -np.inf
    with np.errstate(all="ignore"):
        ref = zo.gemm(a, b, None, 1.0, 1.0, False, False)
    y = torch.zeros((1, 1, 70, 68), device="cuda:0")
    G.tm.gemm_lean(G.dev(a), G.dev(b), None, 1.0, 1.0, False, False, y)
    y = G.host(y)
    np.testing.assert_array_equal(np.isnan(y), np.isnan(ref))
    np.testing.assert_array_equal(np.isposinf(y), np.isposinf(ref))
    np.testing.assert_array_equal(np.isneginf(y), np.isneginf(ref))
    fine = np.isfinite(ref)
    np.testing.assert_allclose(y[fine], ref[fine], rtol=G.RTOL, atol=G.ATOL)


def test_gemm_cut_k_calls_in_a_row_share_nothing(G):
    """Different shapes back to back without a wait: each finds the counters as it needs them."""
    outs = []
    for M, K, N in SHAPES * 3:
        a, b = _inputs(M, K, N)
        y = torch.full((1, 1, M, N), float("nan"), device="cuda:0")
        G.tm.gemm_lean(G.dev(a), G.dev(b), None, 1.0, 1.0, False, False, y)
        outs.append((y, a, b))
    for y, a, b in outs:
        np.testing.assert_allclose(G.host(y)[0, 0], a[0, 0].astype(np.float64) @ b[0, 0].astype(np.float64), rtol=1e-4, atol=2e-5)
