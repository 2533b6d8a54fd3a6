"""3x3 int8 layers of up to 16 channels (two taps of a filter row an operand, the fourth tap's weights zero): channels from 5 to 16, strides,
dilations up to wider than the map's padding, pads that leave the last tap outside, ragged maps, both layouts, with and without a fused
pool.  Bit for bit against the oracle; 17 channels take the other form."""
import numpy as np
import pytest

from oracle import oracle as zo

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import gpu_util
    return gpu_util


def _layer(N, C, H, W, K, seed):
    g = np.random.default_rng(seed)
    return (g.integers(0, 256, (N, C, H, W), dtype=np.uint8), g.integers(-127, 128, (K, C, 3, 3), dtype=np.int8),
            (g.uniform(0.5, 1.5, K) * 0.05 / np.sqrt(9 * C)).astype(np.float32), g.integers(-1000, 1001, K).astype(np.int32))


@pytest.mark.parametrize("act", ["leaky", None])
@pytest.mark.parametrize("N,C,H,W,K,strides,pads,dil", [
    (2, 16, 13, 11, 32, [1, 1], [1, 1, 1, 1], [1, 1]), (3, 5, 9, 17, 7, [1, 1], [0, 0, 0, 0], [1, 1]), (5, 9, 24, 24, 96, [2, 2], [1, 1, 1, 1], [1, 1]),
    (4, 15, 12, 14, 33, [1, 2], [0, 1, 1, 0], [1, 1]), (2, 16, 21, 19, 20, [1, 1], [2, 2, 2, 2], [2, 2]), (2, 12, 16, 23, 64, [1, 1], [1, 3, 1, 3], [1, 5]),
    (300, 16, 6, 6, 16, [1, 1], [1, 1, 1, 1], [1, 1]), (64, 8, 3, 3, 40, [1, 1], [1, 1, 1, 1], [1, 1]), (2, 17, 13, 11, 32, [1, 1], [1, 1, 1, 1], [1, 1])])
def test_layers_match_the_oracle(G, N, C, H, W, K, strides, pads, dil, act):
    x, w, ws, b = _layer(N, C, H, W, K, N + C + K)
    kw = dict(act=act, act_alpha=0.1, act_scale=0.04, act_zp=30) if act else {}
    ref = zo.qlinearconv(x, 0.02, 117, w, ws, None, 0.05, 120, b, strides, pads, dil, 1, **kw)
    y = G.tm.qlinearconv(G.dev(x), 0.02, 117, G.dev(w), G.dev(ws), None, 0.05, 120, G.dev(b), strides, pads, dil, 1, **kw)
    name = G.tm.context().kernel_name()
    assert name.startswith("qconv_mfma_kernel<") and (name.split(",")[3] == "6") == (C <= 16), name
    np.testing.assert_array_equal(G.host(y), ref)


@pytest.mark.parametrize("N,C,H,W,K", [(2, 16, 48, 48, 32), (3, 10, 14, 22, 96), (700, 16, 6, 8, 17)])
def test_between_blocked_tensors_with_a_pool(G, N, C, H, W, K):
    from zant_amd.model import Model, U8
    x, w0, ws0, b0 = _layer(N, 3, H, W, C, 1)
    _, w, ws, b = _layer(N, C, 1, 1, K, 2)
    m = Model(G.tm.context())
    t = m.input((N, 3, H, W), U8, 0.02, 117)
    t = m.qlinearconv(t, w0, ws0, b0, 0.05, 128, [1, 1], [1, 1, 1, 1])
    t = m.qlinearconv(t, w, ws, b, 0.05, 128, [1, 1], [1, 1, 1, 1])
    t = m.maxpool(t, [2, 2], [2, 2])
    w1, ws1 = np.ones((16, K, 1, 1), np.int8), np.full(16, 0.01, np.float32)  # (a pool is fused where what follows reads a blocked tensor)
    t = m.qlinearconv(t, w1, ws1, None, 0.5, 0, [1, 1], [0, 0, 0, 0])
    m.finalize()
    m.profile()
    assert any(k.startswith("qconv_mfma_kernel<") and ",6," in k for k in m.launch_kernels()), m.launch_kernels()
    r = zo.qlinearconv(x, 0.02, 117, w0, ws0, None, 0.05, 128, b0, [1, 1], [1, 1, 1, 1], [1, 1], 1)
    r = zo.qlinearconv(r, 0.05, 128, w, ws, None, 0.05, 128, b, [1, 1], [1, 1, 1, 1], [1, 1], 1)
    r = zo.onnx_maxpool(r, [2, 2], [2, 2], [1, 1], [0, 0, 0, 0])
    r = zo.qlinearconv(r, 0.05, 128, w1, ws1, None, 0.5, 0, None, [1, 1], [0, 0, 0, 0], [1, 1], 1)
    np.testing.assert_array_equal(m.predict_host(x), r)
    m.close()
