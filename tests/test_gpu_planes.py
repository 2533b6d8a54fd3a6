"""Operators on planes whose sizes are not whole vectors: means, batch normalisation, 2x2 pooling, f32 and u8."""
import numpy as np
import pytest
import torch

from oracle import oracle as zo

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import gpu_util
    return gpu_util


# runs of 15 (four lanes), 16 and 63 (sixteen), 64, 256, 257, 512 (a wave, elements), 513 (the general kernel), 516, 764 and 768 (vectors),
# 772 (the general kernel again); 1, 4, 5 and 16 k results and one more: partial groups of four, waves and workgroups
@pytest.mark.parametrize("run", [15, 16, 63, 64, 65, 192, 255, 256, 257, 260, 511, 512, 513, 516, 764, 768, 772])
@pytest.mark.parametrize("rows", [1, 4, 5, 16, 65, 515])
def test_mean_of_planes(G, rows, run):
    x = torch.randn(rows, run, device="cuda", generator=torch.Generator("cuda").manual_seed(rows * 1000 + run)) + 0.5
    y = G.tm.reduce_mean(x, [1], False, False)
    # a sum of n terms, each partial sum rounded once: less than (n / 16 + 16) * 2^-24 of the sum of magnitudes
    bound = (run / 16 + 16) * 2.0 ** -24 * x.double().abs().mean(1)
    assert ((y.double() - x.double().mean(1)).abs() <= bound).all()


def test_mean_of_planes_keeps_infinities_and_nan_to_their_plane(G):
    x = torch.ones(37, 169, device="cuda")
    x[3, 168] = float("inf")
    x[4, 0] = float("nan")
    x[20] = -0.0
    y = G.tm.reduce_mean(x.view(37, 13, 13), [1, 2], False, False).cpu().numpy()
    want = np.ones(37, np.float32)
    want[3], want[4], want[20] = np.inf, np.nan, 0.0
    np.testing.assert_array_equal(y, want)
    assert not np.signbit(y[20])


@pytest.mark.parametrize("shape", [(2, 3, 4), (3, 5, 5), (1, 1, 6), (2, 7, 3), (5, 1, 7), (4, 3, 13, 13), (3, 50, 27, 27), (9, 2, 4099), (7, 5, 9)])
def test_batchnorm_of_planes_that_end_inside_a_vector(G, shape):
    g = torch.Generator("cuda").manual_seed(sum(shape))
    F = shape[1]
    x = torch.randn(shape, device="cuda", generator=g)
    gamma, beta, mean = (torch.randn(F, device="cuda", generator=g) for _ in range(3))
    var = torch.rand(F, device="cuda", generator=g) + 0.1
    y = G.tm.batchnorm(x, gamma, beta, mean, var, 1e-5)
    s = (1, F) + (1,) * (len(shape) - 2)
    centred = (x - mean.view(s)).double()
    scaled = centred / (var + 1e-5).double().sqrt().view(s) * gamma.double().view(s)
    # root, quotient, product and sum are rounded once each: half a unit in the last place of each step's result
    bound = 2.0 ** -24 * (4 * scaled.abs() + (scaled + beta.double().view(s)).abs())
    assert ((y.double() - scaled - beta.double().view(s)).abs() <= bound).all()


@pytest.mark.parametrize("shape", [(1, 1, 4, 5), (2, 3, 5, 5), (3, 7, 13, 11), (2, 4, 4, 255), (1, 5, 31, 33), (2, 3, 64, 65), (5, 1, 27, 27)])
def test_pools_of_planes_of_odd_width(G, shape):
    x = torch.randn(shape, device="cuda", generator=torch.Generator("cuda").manual_seed(shape[3]))
    x[0, 0, 0, 0], x[-1, -1, 1, 2] = float("inf"), float("nan")
    w = x[:, :, :shape[2] // 2 * 2, :shape[3] // 2 * 2]
    a, b, c, d = w[:, :, ::2, ::2], w[:, :, ::2, 1::2], w[:, :, 1::2, ::2], w[:, :, 1::2, 1::2]
    np.testing.assert_array_equal(G.host(G.tm.avgpool(x, [2, 2], [2, 2])), (((a + b) + c + d) / 4).cpu().numpy())
    y = G.tm.onnx_maxpool(x, [2, 2], [2, 2], [1, 1], [0, 0, 0, 0])
    np.testing.assert_array_equal(G.host(y), torch.fmax(torch.fmax(a, b), torch.fmax(c, d)).cpu().numpy())


# rows of 3 results (byte by byte), 4 to 7 (vectors of four), 8 up (of eight, the last moved back); odd heights, one row, one plane
@pytest.mark.parametrize("shape", [(2, 3, 5, 7), (1, 1, 2, 8), (3, 2, 7, 9), (2, 5, 6, 15), (1, 1, 2, 16), (2, 3, 9, 17), (3, 7, 13, 11),
                                   (4, 5, 27, 27), (3, 2, 50, 33), (1, 2, 4, 34), (2, 3, 48, 50), (40, 30, 21, 43)])
def test_byte_pools_of_any_width(G, shape):
    x = torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=torch.Generator("cuda").manual_seed(shape[3]))
    w = x[:, :, :shape[2] // 2 * 2, :shape[3] // 2 * 2]
    want = torch.maximum(torch.maximum(w[:, :, ::2, ::2], w[:, :, ::2, 1::2]), torch.maximum(w[:, :, 1::2, ::2], w[:, :, 1::2, 1::2]))
    assert torch.equal(G.tm.onnx_maxpool(x, [2, 2], [2, 2], [1, 1], [0, 0, 0, 0]), want)
    off = torch.cat([x.flatten(), x.flatten()[:3]])[3:].view(shape)  # from an odd address
    assert off.data_ptr() % 4 == 3
    y = torch.zeros(want.numel() + 5, dtype=torch.uint8, device="cuda")
    G.tm.onnx_maxpool_lean(off, y[5:].view(want.shape), [2, 2], [2, 2], [1, 1], [0, 0, 0, 0])
    w = off[:, :, :shape[2] // 2 * 2, :shape[3] // 2 * 2]
    want = torch.maximum(torch.maximum(w[:, :, ::2, ::2], w[:, :, ::2, 1::2]), torch.maximum(w[:, :, 1::2, ::2], w[:, :, 1::2, 1::2]))
    assert torch.equal(y[5:].view(want.shape), want) and not y[:5].any()


@pytest.mark.parametrize("hw", [(1, 1), (3, 5), (4, 4), (1, 17), (7, 7), (8, 8), (5, 13), (13, 13), (31, 33), (32, 32), (25, 41), (57, 55), (90, 91)])
@pytest.mark.parametrize("planes", [1, 3, 17, 260])
def test_byte_means_of_any_plane(G, planes, hw):
    g = np.random.default_rng(planes * 1000 + hw[0] * hw[1])
    x = g.integers(0, 256, (1, planes) + hw, dtype=np.uint8)
    want = zo.qlinear_global_avgpool(x, 0.05, 128, 0.02, 110)
    np.testing.assert_array_equal(G.host(G.tm.qlinear_global_avgpool(G.dev(x), 0.05, 128, 0.02, 110)), want)
    buf = G.dev(np.concatenate([np.zeros(3, np.uint8), x.ravel()]))  # from an odd address
    np.testing.assert_array_equal(G.host(G.tm.qlinear_global_avgpool(buf[3:].view(x.shape), 0.05, 128, 0.02, 110)), want)
