"""Position tables of the fused inverted residual block: tiles of several images of odd and even maps under both strides, the last one partly
filled, rows that do not divide a map, and a block whose weights leave room for a row or two.  Bit for bit against the oracle, layer by layer."""
import numpy as np
import pytest

import int8_ref
from test_gpu_qblock import _arch

pytestmark = pytest.mark.gpu

CASES = [
    # (H, W), stem channels, blocks (hidden, cout, stride, activations, depthwise padding), batch
    ((7, 7), 96, [(576, 96, 1, "relu6", "relu6", 1)], 3),
    ((4, 6), 8, [(48, 16, 2, "relu6", "relu6", 1)], 701),
    ((5, 3), 16, [(64, 24, 2, "relu6", "leaky", 1)], 1027),
    ((6, 5), 40, [(80, 40, 1, "leaky", "relu6", 1)], 515),
    ((11, 30), 24, [(72, 24, 1, "relu6", "relu6", 1)], 2),
    ((23, 9), 20, [(60, 40, 2, "relu6", "relu6", 1)], 5),
]


@pytest.mark.parametrize("hw,c0,blocks,batch", CASES, ids=[str(i) for i in range(len(CASES))])
def test_blocks_match_the_oracle(hw, c0, blocks, batch):
    import gpu_util as G
    from zant_amd import networks as nets
    arch = _arch(hw, c0, blocks)
    params = nets.int8_params(arch, seed=7)
    rng = np.random.default_rng(batch)
    quant = int8_ref.calibrate(arch, params, rng.integers(0, 256, (2,) + arch["input"], dtype=np.uint8))
    x = rng.integers(0, 256, (batch,) + arch["input"], dtype=np.uint8)
    sample = np.unique(np.r_[0:min(batch, 5), max(batch - 5, 0):batch])
    m = nets.build_int8_model(G.tm.context(), arch, params, quant, batch)
    assert m.num_launches == 3
    np.testing.assert_array_equal(m.predict_host(x)[sample], int8_ref.forward(arch, params, quant, x[sample]))
    m.close()


@pytest.mark.parametrize("hw,c0,blocks,batch,kernel", [
    ((4, 4), 40, [(240, 64, 2, "relu6", "relu6", 1)], 256, "qblock_kernel<2,1,true,true>"),   # eight chunks on one position tile: shared
    ((6, 6), 24, [(72, 32, 1, "relu6", "relu6", 1)], 1, "qblock_kernel<1,1,true,true>"),      # three
    ((3, 3), 24, [(72, 40, 2, "relu6", "relu6", 1)], 32, "qblock_kernel<2,1,true,false>"),    # three, two blocks of output channels: not shared
    # patches of many channel blocks, dealt in a row
    ((7, 7), 72, [(72, 72, 1, "relu6", "relu6", 1)], 1030, "qblock_flat_kernel<3,1,true,false>"),
    ((13, 11), 100, [(96, 128, 2, "relu6", "leaky", 1)], 5, "qblock_flat_kernel<4,1,true,false>"),
    ((112, 112), 40, [(120, 40, 1, "relu6", "relu6", 1)], 1, "qblock_flat_kernel<2,1,true,false>"),
    ((4, 4), 96, [(192, 56, 1, "relu6", "relu6", 1)], 2, "qblock_flat_kernel<2,1,true,true>"),
])
def test_few_positions_and_many_channel_blocks(hw, c0, blocks, batch, kernel):
    import gpu_util as G
    from zant_amd import networks as nets
    arch = _arch(hw, c0, blocks)
    params = nets.int8_params(arch, seed=9)
    rng = np.random.default_rng(batch)
    quant = int8_ref.calibrate(arch, params, rng.integers(0, 256, (2,) + arch["input"], dtype=np.uint8))
    x = rng.integers(0, 256, (batch,) + arch["input"], dtype=np.uint8)
    m = nets.build_int8_model(G.tm.context(), arch, params, quant, batch)
    m.profile()
    assert m.launch_kernels()[1] == kernel, m.launch_kernels()
    sample = np.unique(np.r_[0:min(batch, 5), max(batch - 5, 0):batch])
    np.testing.assert_array_equal(m.predict_host(x)[sample], int8_ref.forward(arch, params, quant, x[sample]))
    m.close()
