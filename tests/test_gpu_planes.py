"""The mean of planes whose sizes are not whole vectors, few loads a lane."""
import numpy as np
import pytest
import torch

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
