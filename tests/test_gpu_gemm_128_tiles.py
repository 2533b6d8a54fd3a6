"""The f32 Gemm's 128x128 tiles, whose eight waves all multiply and stage: sums around a step of 32 terms, around the six steps its loop
runs through, and that end inside a step, where the last 32 terms are taken again with zeros; every storage order, ragged edges."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import gpu_util
    return gpu_util


def _gemm(G, M, K, N, ta, tb, spoil=None):
    g = torch.Generator("cuda").manual_seed(M + K + N)
    a, b = torch.randn(M, K, device="cuda", generator=g), torch.randn(K, N, device="cuda", generator=g) * K ** -0.5
    c = torch.randn(1, 1, 1, N, device="cuda", generator=g)
    if spoil:
        spoil(a, b)
    A, B = (a.t() if ta else a).contiguous().view(1, 1, *((K, M) if ta else (M, K))), (b.t() if tb else b).contiguous()
    y = torch.full((1, 1, M, N), float("nan"), device="cuda")
    G.tm.gemm_lean(A, B.view(1, 1, *B.shape), c, 1.0, 1.0, ta, tb, y, None)
    assert G.tm.context().kernel_name().startswith("gemm_f32_split_kernel<2,2,3,"), G.tm.context().kernel_name()
    return a, b, c, y[0, 0]


@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("K", [97, 127, 128, 129, 159, 160, 161, 191, 192, 193, 224, 225, 257, 997])  # (shorter sums are other tiles')
def test_sums_of_few_steps(G, K, ta, tb):
    M, N = 8189, 1021
    a, b, c, y = _gemm(G, M, K, N, ta, tb)
    want = a.double() @ b.double() + c[0, 0].double()
    rms = want.square().mean().sqrt()
    # K products of unit variance over K, each partial sum rounded once in f32
    assert (y.double() - want).square().mean().sqrt() < K ** 0.5 * 2.0 ** -24 * rms
    assert (y.double() - want).abs().max() < 8 * K ** 0.5 * 2.0 ** -24 * rms + 2.0 ** -24 * want.abs().max()


@pytest.mark.parametrize("K", [101, 256])
def test_an_infinity_and_a_nan_stay_in_their_rows_and_columns(G, K):
    def spoil(a, b):
        a[5, K - 1], a[130, 0], a[200, 66] = float("inf"), float("nan"), 3e38
        b[70, 9] = float("-inf")  # (a term that a last step inside K takes again)
    a, b, c, y = _gemm(G, 8189, K, 1021, False, True, spoil)
    want = (a.double() @ b.double() + c[0, 0].double()).float()
    clean = torch.isfinite(want)
    assert torch.equal(torch.isnan(y), torch.isnan(want)) and torch.equal(torch.isinf(y), torch.isinf(want))
    assert (y[clean] - want[clean]).abs().div(want[clean].abs() + 1).max() < 1e-5
