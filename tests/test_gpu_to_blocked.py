"""The change of layout NCHW u8 -> 16-channel blocks at planes of any length and any address, alone and in the launch that also packs a
convolution's weights."""
import numpy as np
import pytest
import torch

from oracle import oracle as zo

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import gpu_util
    return gpu_util


# planes of 1 to 9 positions, a quad past whole workgroups of 64 quads, channels around a block, an address that is no multiple of 4
@pytest.mark.parametrize("off", [0, 1, 3])
@pytest.mark.parametrize("N,C,H,W", [(3, 1, 1, 1), (2, 17, 1, 2), (3, 16, 1, 3), (5, 33, 2, 2), (2, 15, 5, 1), (7, 19, 1, 7), (4, 32, 3, 3),
                                     (2, 5, 16, 16), (3, 20, 17, 15), (9, 40, 23, 11)])
def test_to_blocked_any_plane(G, N, C, H, W, off):
    x = np.random.default_rng(N + C + H * W).integers(0, 256, (N, C, H, W), dtype=np.uint8)
    flat = torch.zeros(x.size + 8, dtype=torch.uint8, device="cuda:0")
    X = flat[off:off + x.size].view(x.shape)
    X.copy_(torch.from_numpy(x))
    xb = G.host(G.tm.to_blocked16(X)).reshape(N, (C + 15) // 16, H, W, 16)
    want = np.full((N, (C + 15) // 16 * 16, H, W), 0x80, np.uint8)  # (channels past C: the kernel writes zeros)
    want[:, :C] = x
    np.testing.assert_array_equal(xb ^ 0x80, want.reshape(N, -1, 16, H, W).transpose(0, 1, 3, 4, 2))


# the tiled, the patch-stationary and the depthwise kernel, whose weights are packed in the launch that blocks their input
@pytest.mark.parametrize("N,C,H,W,K,ks,pad,group", [(5, 19, 7, 9, 40, 1, 0, 1), (3, 40, 13, 11, 70, 3, 1, 1), (4, 33, 15, 9, 33, 3, 1, 33),
                                                    (30, 8, 3, 3, 9, 3, 1, 1), (70, 48, 1, 1, 50, 1, 0, 1)])
def test_qconv_with_its_packing_and_layout_in_one_launch(G, N, C, H, W, K, ks, pad, group):
    g = np.random.default_rng(N + C + K)
    x = g.integers(0, 256, (N, C, H, W), dtype=np.uint8)
    w = g.integers(-127, 128, (K, C // group, ks, ks), dtype=np.int8)
    ws = g.uniform(0.0005, 0.002, K).astype(np.float32)
    b = g.integers(-500, 500, K, dtype=np.int32)
    args = ([1, 1], [pad] * 4, [1, 1], group)
    ref = zo.qlinearconv(x, 0.02, 131, w, ws, None, 0.05, 120, b, *args)
    y = torch.zeros(ref.shape, dtype=torch.uint8, device="cuda:0")
    G.tm.qlinearconv_lean(G.dev(x), 0.02, 131, G.dev(w), G.dev(ws), None, 0.05, 120, G.dev(b), y, *args, "none", 0.0, 0.05, 120)
    np.testing.assert_array_equal(G.host(y), ref)
