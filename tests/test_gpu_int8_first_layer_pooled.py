"""First layers of up to 16 filters with a 2x2 pool behind them (a window's left and right member from one chain of matrix instructions):
numbers of filters around the 8 and 16 rows, every number of channels, odd rows and columns, pads, negative scales (the window's lowest
accumulator instead of its highest), one image and many.  Bit for bit against the oracle; 17 filters take the wider form."""
import numpy as np
import pytest

from oracle import oracle as zo

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import gpu_util
    return gpu_util


@pytest.mark.parametrize("act", ["leaky", None])
@pytest.mark.parametrize("N,C,H,W,K,pads", [
    (1, 3, 6, 6, 16, [1, 1, 1, 1]), (2, 1, 7, 9, 1, [1, 1, 1, 1]), (3, 4, 10, 13, 8, [1, 1, 1, 1]), (2, 2, 9, 8, 9, [0, 0, 0, 0]),
    (40, 3, 12, 11, 15, [1, 1, 1, 1]), (5, 3, 33, 34, 16, [0, 1, 1, 0]), (3, 3, 14, 14, 17, [1, 1, 1, 1]), (700, 1, 4, 4, 4, [1, 1, 1, 1])])
def test_pooled_first_layer(G, N, C, H, W, K, pads, act):
    from zant_amd.model import Model, U8
    g = np.random.default_rng(N + 10 * C + K)
    x = g.integers(0, 256, (N, C, H, W), dtype=np.uint8)
    w = g.integers(-127, 128, (K, C, 3, 3), dtype=np.int8)
    ws = (g.uniform(0.5, 1.5, K) * 0.05 / np.sqrt(9 * C)).astype(np.float32)
    ws[::3] *= -1  # a negative multiplier turns the order of the accumulators round
    b = g.integers(-1000, 1001, K).astype(np.int32)
    m = Model(G.tm.context())
    t = m.input((N, C, H, W), U8, 0.02, 117)
    t = m.qlinearconv(t, w, ws, b, 0.05, 128, [1, 1], pads)
    if act:
        t = m.qlinear_act(t, act, 0.1, 0.04, 30)
    t = m.maxpool(t, [2, 2], [2, 2])
    m.finalize()
    m.profile()
    want = f"qfirst_mfma_kernel<{C},1,true,{8 if K <= 16 else 16}>"
    assert want in m.launch_kernels(), m.launch_kernels()
    r = zo.qlinearconv(x, 0.02, 117, w, ws, None, 0.05, 128, b, [1, 1], pads, [1, 1], 1)
    if act:
        r = zo.qlinear_act(r, 0.05, 128, act, 0.1, 0.04, 30)
    np.testing.assert_array_equal(m.predict_host(x), zo.onnx_maxpool(r, [2, 2], [2, 2], [1, 1], [0, 0, 0, 0]))
    m.close()
