"""The matrix-core f32 convolution and Gemm split their operands into bf16 terms: over the whole range of f32, subnormal numbers
included, the result has to stay as close to 64 bits as f32 sums are."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import gpu_util
    return gpu_util


def _scaled(g, shape, exponent):
    return (g.standard_normal(shape) * 2.0 ** exponent).astype(np.float32)


def _check(y, ref, terms, exponent):
    """f32 sums of `terms` products are a random walk of roundings: below sqrt(terms) * 2^-24 of the result's root mean square,
    plus the rounding of a subnormal result (half of 2^-149) where the products lie that low."""
    rms = np.sqrt(np.mean(ref ** 2))
    assert rms > 0
    err = np.sqrt(np.mean((y.astype(np.float64) - ref) ** 2))
    assert err < np.sqrt(terms) * 2.0 ** -24 * rms + 2.0 ** -150, (exponent, err / rms)


# one operand's exponent and the other's: both directions, down to single-bit subnormal numbers, and up to sums near overflow
EXPONENTS = [(-112, 0), (-118, 60), (-126, 0), (-130, 100), (-140, 120), (-147, 110), (0, -126), (90, -140), (-60, -60), (110, 3), (8, 100)]


@pytest.mark.parametrize("ea,eb", EXPONENTS)
@pytest.mark.parametrize("tb", [False, True])
def test_gemm_over_the_exponent_range(G, ea, eb, tb):
    import torch
    g = np.random.default_rng(abs(ea) + 7 * abs(eb))
    M, K, N = 70, 100, 66
    a, b = _scaled(g, (1, 1, M, K), ea), _scaled(g, (1, 1, K, N), eb)
    y = torch.full((1, 1, M, N), float("nan"), device="cuda:0")
    G.tm.gemm_lean(G.dev(a), G.dev(np.swapaxes(b, -1, -2).copy() if tb else b), None, 1.0, 1.0, False, tb, y)
    assert G.tm.context().kernel_name().startswith("gemm_f32_split_kernel<")
    _check(G.host(y)[0, 0], a[0, 0].astype(np.float64) @ b[0, 0].astype(np.float64), K, (ea, eb))


@pytest.mark.parametrize("ea,eb", EXPONENTS)
@pytest.mark.parametrize("C,k", [(20, 3), (12, 3), (40, 1)])  # whole-step channels, two taps per instruction, 1x1
def test_conv_over_the_exponent_range(G, ea, eb, C, k):
    g = np.random.default_rng(abs(ea) + 7 * abs(eb) + C)
    x, w = _scaled(g, (2, C, 11, 13), ea), _scaled(g, (33, C, k, k), eb)
    y = G.host(G.tm.Conv(G.dev(x), G.dev(w), None, [1, 1], [0, 0, 0, 0], [1, 1], 1, "NOTSET"))
    assert G.tm.context().kernel_name().startswith("conv_f32_split_kernel<")
    win = np.lib.stride_tricks.sliding_window_view(x.astype(np.float64), (k, k), axis=(2, 3))
    _check(y, np.einsum("nchwij,kcij->nkhw", win, w.astype(np.float64)), C * k * k, (ea, eb))
