"""Fully connected int8 layers of few images (a wave an output channel) and where other kernels are faster: numbers of images around the
groups of four and the limit of 64, channels around a wave's 1024, output channels that leave waves or a blocked tensor's last block empty,
both layouts, activations.
Bit for bit against the oracle; what the kernel does not take gives the same."""
import numpy as np
import pytest

from oracle import oracle as zo

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import gpu_util
    return gpu_util


def _layer(N, C, K, seed):
    g = np.random.default_rng(seed)
    return (g.integers(0, 256, (N, C, 1, 1), dtype=np.uint8), g.integers(-127, 128, (K, C, 1, 1), dtype=np.int8),
            (g.uniform(0.5, 1.5, K) * 0.05 / np.sqrt(C)).astype(np.float32), g.integers(-1000, 1001, K).astype(np.int32))


@pytest.mark.parametrize("act", ["none", "leaky", "relu6"])
@pytest.mark.parametrize("N,C,K", [(1, 16, 1), (1, 1280, 1000), (1, 2048, 1024), (3, 48, 5), (4, 1008, 4), (5, 1024, 3), (7, 1040, 33), (33, 2064, 17), (63, 4096, 9),
                                   (64, 3072, 30), (65, 1280, 12), (2, 4112, 7), (9, 40, 21),
                                   # many filters: on the matrix cores, past what these have room for here again, of few terms the direct kernel
                                   (64, 64, 4096), (40, 256, 4096), (40, 16, 8192)])
def test_layers_match_the_oracle(G, N, C, K, act):
    x, w, ws, b = _layer(N, C, K, N + C + K)
    y = G.dev(np.full((N, K, 1, 1), 77, np.uint8))
    G.tm.qlinearconv_lean(G.dev(x), 0.02, 117, G.dev(w), G.dev(ws), None, 0.05, 128, G.dev(b), y, [1, 1], [0] * 4, [1, 1], 1, act, 0.1, 0.04, 30)
    here = N <= 64 and C % 16 == 0 and C <= 4096 and (N, C, K) not in ((64, 64, 4096), (40, 16, 8192))
    assert G.tm.context().kernel_name().startswith("qfc_kernel<") == here, G.tm.context().kernel_name()
    want = zo.qlinearconv(x, 0.02, 117, w, ws, None, 0.05, 128, b, [1, 1], [0] * 4, [1, 1], 1)
    if act != "none":
        want = zo.qlinear_act(want, 0.05, 128, act, 0.1, 0.04, 30)
    np.testing.assert_array_equal(G.host(y), want)


def test_without_bias_and_with_one_scale(G):
    x, w, ws, b = _layer(6, 256, 10, 3)
    y = G.dev(np.zeros((6, 10, 1, 1), np.uint8))
    G.tm.qlinearconv_lean(G.dev(x), 0.02, 0, G.dev(w), G.dev(ws[:1]), None, 0.05, 3, None, y, [1, 1], [0] * 4, [1, 1], 1)
    np.testing.assert_array_equal(G.host(y), zo.qlinearconv(x, 0.02, 0, w, ws[:1], None, 0.05, 3, None, [1, 1], [0] * 4, [1, 1], 1))


def test_operands_off_16_bytes_take_another_kernel(G):
    import torch
    x, w, ws, b = _layer(2, 64, 5, 4)
    flat = torch.zeros(x.size + 16, dtype=torch.uint8, device="cuda")
    X = flat[1:1 + x.size].view(2, 64, 1, 1)
    X.copy_(torch.from_numpy(x))
    y = G.dev(np.zeros((2, 5, 1, 1), np.uint8))
    G.tm.qlinearconv_lean(X, 0.02, 117, G.dev(w), G.dev(ws), None, 0.05, 128, G.dev(b), y, [1, 1], [0] * 4, [1, 1], 1)
    assert not G.tm.context().kernel_name().startswith("qfc_kernel<")
    np.testing.assert_array_equal(G.host(y), zo.qlinearconv(x, 0.02, 117, w, ws, None, 0.05, 128, b, [1, 1], [0] * 4, [1, 1], 1))


@pytest.mark.parametrize("N", [1, 5, 64])
def test_chained_in_a_model(G, N):
    """Blocked in and out between two such layers of a model, the last block of 16 channels partly padding."""
    from zant_amd.model import Model, U8
    layers = [_layer(N, 96, 40, 5), _layer(N, 40, 48, 6), _layer(N, 48, 33, 7), _layer(N, 33, 10, 8)]
    m = Model(G.tm.context())
    t = m.input((N, 96, 1, 1), U8, 0.02, 128)
    v = layers[0][0]
    x, s, z = v, 0.02, 128
    for _, w, ws, b in layers:
        t = m.qlinearconv(t, w, ws, b, 0.05, 120, [1, 1], [0] * 4, [1, 1], 1)
        v, s, z = zo.qlinearconv(v, s, z, w, ws, None, 0.05, 120, b, [1, 1], [0] * 4, [1, 1], 1), 0.05, 120
    m.finalize()
    m.profile()
    # 48 channels in, and 96; of 64 images, with the weights kept, the matrix-core kernel is the faster one
    assert sum(k.startswith("qfc_kernel<") for k in m.launch_kernels()) == (2 if N < 64 else 0), m.launch_kernels()
    np.testing.assert_array_equal(m.predict_host(x), v)
    m.close()
