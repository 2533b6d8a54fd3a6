"""The matrix-core f32 convolution of short sums (operands gathered from memory) where its tiling can go wrong: groups of terms that
do not fill, blocks of channels that do not fill, tiles that span many images, padding on every side, more terms than one workgroup's
usual share of LDS, and operands at the ends of the f32 range."""
import numpy as np
import pytest

from oracle import oracle as zo

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import gpu_util
    return gpu_util


CASES = [
    # N, C, H, W, K, (KH, KW), stride, dilation, pads
    (3, 1, 9, 7, 5, (3, 3), 1, 1, [1, 1, 1, 1]),         # 9 terms: half a group and a lone last one
    (2, 3, 23, 31, 33, (5, 5), 1, 1, [2, 2, 2, 2]),      # 75 terms, filters one past a block
    (1, 2, 40, 33, 97, (3, 3), 2, 1, [1, 0, 2, 1]),      # 18 terms in chunks of 8, four blocks, uneven padding, stride 2
    (70, 3, 4, 4, 8, (3, 3), 1, 1, [0, 0, 0, 0]),        # four positions an image: a tile spans nine of them
    (2, 31, 19, 17, 70, (1, 1), 1, 1, [0, 0, 0, 0]),     # 31 terms
    (400, 32, 19, 17, 96, (1, 1), 2, 1, [0, 0, 0, 0]),     # 32 terms, three blocks a workgroup
    (110, 40, 19, 17, 64, (1, 1), 1, 1, [0, 0, 0, 0]),    # two blocks a workgroup, chunks of 16 and a half one
    (1, 3, 30, 30, 40, (11, 11), 1, 2, [10, 10, 10, 10]),  # 363 terms, dilated, padding wider than the tile's halo
    (3, 6, 11, 13, 20, (3, 3), 1, 1, [1, 1, 1, 1]),      # few positions: taken from the split kernel
    (300, 2, 26, 26, 3, (1, 2), 1, 1, [0, 0, 0, 1]),     # 4 terms, more tiles than waves
]


@pytest.mark.parametrize("case", CASES, ids=[str(i) for i in range(len(CASES))])
@pytest.mark.parametrize("relu", [False, True])
def test_conv_short_tilings_vs_oracle(G, case, relu):
    N, C, H, W, K, (kh, kw), s, d, pads = case
    g = np.random.default_rng(N + C + K)
    x = g.standard_normal((N, C, H, W), dtype=np.float32)
    w = (g.standard_normal((K, C, kh, kw)) * np.sqrt(2.0 / (C * kh * kw))).astype(np.float32)
    b = (g.standard_normal(K) * 0.1).astype(np.float32)
    args = ([s, s], pads, [d, d], 1, "NOTSET")
    pick = list(range(N)) if N <= 8 else [0, 1, N // 2, N - 1]
    ref = zo.Conv(x[pick], w, b, *args)
    shape = G.tm.get_convolution_output_shape(x.shape, w.shape, [s, s], pads, [d, d], "NOTSET")
    y = G.dev(np.full(shape, np.nan, np.float32))
    G.tm.conv_lean(G.dev(x), G.dev(w), y, G.dev(b), *args, fuse_act="relu" if relu else None)
    assert G.tm.context().kernel_name().startswith("conv_f32_short_kernel<"), G.tm.context().kernel_name()
    np.testing.assert_allclose(G.host(y)[pick], zo.ReLU(ref) if relu else ref, rtol=G.RTOL, atol=G.ATOL)


@pytest.mark.parametrize("terms", [5, 17, 32, 100])
def test_conv_short_is_as_close_to_64_bits_as_f32_sums(G, terms):
    """Sums of `terms` products of normal operands: a random walk of roundings stays below sqrt(terms) * 2^-24 * the result's root
    mean square (every partial sum is at most the result's size, in the mean)."""
    g = np.random.default_rng(terms)
    x = g.standard_normal((4, terms, 60, 50), dtype=np.float32)
    w = g.standard_normal((64, terms, 1, 1)).astype(np.float32)
    y = G.host(G.tm.Conv(G.dev(x), G.dev(w), None, [1, 1], [0, 0, 0, 0], [1, 1], 1, "NOTSET"))
    assert G.tm.context().kernel_name().startswith("conv_f32_short_kernel<")
    ref = np.einsum("nchw,kc->nkhw", x.astype(np.float64), w[:, :, 0, 0].astype(np.float64))
    assert np.sqrt(np.mean((y - ref) ** 2)) < np.sqrt(terms) * 2.0 ** -24 * np.sqrt(np.mean(ref ** 2))


def test_conv_short_range_of_operands(G):
    """Subnormal, huge, infinite and NaN operands give what f32 arithmetic gives; padding is zero also beside infinities."""
    g = np.random.default_rng(9)
    x = g.standard_normal((4, 3, 16, 16), dtype=np.float32)
    x[1] *= np.float32(2.0 ** -130)
    x[2] *= np.float32(2.0 ** 125)
    x[3, 0, 0, 0], x[3, 1, 8, 8] = np.inf, np.nan
    w = (np.abs(g.standard_normal((40, 3, 5, 5))) * 0.01).astype(np.float32)
    w[:, :, ::2, ::2] = 0
    args = ([1, 1], [2, 2, 2, 2], [1, 1], 1, "NOTSET")
    with np.errstate(all="ignore"):
        ref = zo.Conv(x, w, None, *args)
    y = G.host(G.tm.Conv(G.dev(x), G.dev(w), None, *args))
    assert G.tm.context().kernel_name().startswith("conv_f32_short_kernel<")
    np.testing.assert_array_equal(np.isnan(y), np.isnan(ref))
    np.testing.assert_array_equal(np.isposinf(y), np.isposinf(ref))
    fine = np.isfinite(ref)
    assert not fine[3].all() and fine[:3].all()
    np.testing.assert_allclose(y[0], ref[0], rtol=G.RTOL, atol=G.ATOL)
    np.testing.assert_allclose(y[1], ref[1], rtol=G.RTOL, atol=75 * 2.0 ** -149)  # a term may round to a multiple of 2^-149
    np.testing.assert_allclose(y[2], ref[2], rtol=G.RTOL, atol=G.ATOL * 2.0 ** 125)
