"""Requantisation by rounding to the address of a table's entry, in the inverted residual block's kernels: zero points of either
parity (a tie goes to the even neighbour of the value without its zero point), tables that change over all, few or none of their
entries, sums far outside the bytes' range, multipliers that put sums on ties.  Bit for bit against the oracle's layers."""
import numpy as np
import pytest

from oracle import oracle as zo

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import gpu_util
    return gpu_util


#        zero points of the two convolutions, activation, its scale and zero point, weight scales, largest bias
CASES = [(127, 128, "relu6", 0.03, 0, (0.001, 0.004), 100),
         (128, 1, "relu6", 0.03, 3, (0.001, 0.004), 100),
         (255, 0, "leaky", 0.05, 77, (0.001, 0.004), 100),      # every entry of its own / ends of the range
         (64, 201, "leaky", 0.011, 131, (0.001, 0.004), 100),   # a table that saturates at both ends
         (13, 14, "relu6", 9.0, 5, (0.001, 0.004), 100),        # a table of two values
         (13, 14, "relu6", 1000.0, 5, (0.001, 0.004), 100),     # a constant table
         (101, 102, "relu6", 0.03, 0, (3.0, 9.0), 100),         # multipliers above 2
         (101, 102, "leaky", 0.03, 9, (1e-9, 1e-3), 2 ** 30),   # sums of 2^30
         (99, 100, "leaky", 0.02, 50, (0.125, 0.125), 50),      # x_scale / y_scale * 0.125 a power of two: ties
         (100, 99, "leaky", 0.02, 50, (0.125, 0.125), 50)]


@pytest.mark.parametrize("N,H,stride", [(2, 14, 1), (600, 6, 1), (3, 9, 2)])
@pytest.mark.parametrize("zp1,zp2,act,a_scale,a_zp,ws_range,bias", CASES)
def test_block_requantisation(G, zp1, zp2, act, a_scale, a_zp, ws_range, bias, N, H, stride):
    from zant_amd.model import Model, U8
    g = np.random.default_rng(zp1 * 256 + zp2 + N)
    m = Model(G.tm.context())
    Cin, Ce, Co = 16, 48, 16
    t = m.input((N, Cin, H, H), U8, 0.5, 128)
    layers = []

    def conv(t, cin, cout, k, s, grp, zp, act):
        w = g.integers(-127, 128, (cout, cin // grp, k, k), dtype=np.int8)
        ws = g.uniform(*ws_range, cout).astype(np.float32)
        b = g.integers(-bias, bias + 1, cout).astype(np.int32)
        layers.append((w, ws, b, s, k // 2, grp, zp, act))
        t = m.qlinearconv(t, w, ws, b, 0.5, zp, [s, s], [k // 2] * 4, [1, 1], grp)
        return m.qlinear_act(t, act, 0.1, a_scale, a_zp) if act else t

    t = conv(t, Cin, Cin, 1, 1, 1, 128, None)
    for _ in range(2):  # two blocks: a chain where the batch allows one
        t = conv(t, Cin, Ce, 1, 1, 1, zp1, act)
        t = conv(t, Ce, Ce, 3, stride, Ce, zp2, act)
        t = conv(t, Ce, Co, 1, 1, 1, 128, None)
    conv(t, Co, Co, 1, 1, 1, 128, None)
    m.finalize()
    assert any("InvertedResidual" in p[0] for p in m.profile())
    x = g.integers(0, 256, (N, Cin, H, H), dtype=np.uint8)
    y = m.predict_host(x)
    m.close()
    sample = np.unique(np.r_[0:min(N, 2), N - 1])
    v, sc, zp = x[sample], 0.5, 128
    for w, ws, b, s, p, grp, z, a in layers:
        v, sc, zp = zo.qlinearconv(v, sc, zp, w, ws, None, 0.5, z, b, [s, s], [p] * 4, [1, 1], grp), 0.5, z
        if a:
            v, sc, zp = zo.qlinear_act(v, sc, zp, a, 0.1, a_scale, a_zp), a_scale, a_zp
    np.testing.assert_array_equal(y[sample], v)
