"""The Gemm of at most sixteen columns: stages of 512 k that end inside a lane's loads, rows and columns short of a tile."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import gpu_util
    return gpu_util


def gemm(G, a, b, c, tb):
    return G.tm.gemm(a[None, None], b[None, None], c[None, None], 1.0, 1.0, False, tb)[0, 0]


@pytest.mark.parametrize("tb", [False, True])
@pytest.mark.parametrize("m,n", [(1, 1), (3, 10), (16, 16), (17, 5), (401, 12)])
@pytest.mark.parametrize("k", [1, 15, 16, 17, 63, 65, 500, 511, 512, 513, 1024, 1300])
def test_gemm_of_few_columns(G, k, m, n, tb):
    g = torch.Generator("cuda").manual_seed(k * 100 + n)
    a = torch.randn(m, k, device="cuda", generator=g)
    b = torch.randn((n, k) if tb else (k, n), device="cuda", generator=g)
    c = torch.randn(1, n, device="cuda", generator=g)
    y = gemm(G, a, b, c, tb)
    bk = (b.t() if tb else b).double()
    # a lane's chain of ceil(k / 64) products and six exchanges, then the bias: one rounding each, of at most the sum of magnitudes
    bound = ((k + 63) // 64 + 8) * 2.0 ** -24 * (a.double().abs() @ bk.abs() + c.abs())
    assert ((y.double() - (a.double() @ bk + c)).abs() <= bound).all()


@pytest.mark.parametrize("k", [5, 70, 700])
def test_gemm_of_few_columns_keeps_infinities(G, k):
    a, b = torch.ones(3, k, device="cuda"), torch.ones(k, 4, device="cuda")
    a[1, k - 1] = float("inf")
    b[k - 1, 2] = float("inf")
    y = gemm(G, a, b, torch.zeros(1, 4, device="cuda"), False)
    want = torch.full((3, 4), float(k), device="cuda")
    want[1], want[:, 2] = float("inf"), float("inf")
    assert torch.equal(y, want)
