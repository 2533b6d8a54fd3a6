"""Chains of inverted residual blocks on one image a workgroup, activations in LDS from block to block: maps of odd sizes under both
strides, one to four blocks of 32 output channels, more units than waves and fewer, and weights that do not fit beside the running
block's.  Each chain is checked against the oracle, block by block, as the chains of several images a workgroup are."""
import pytest

from test_gpu_int8_block import test_blocks_in_a_row_run_as_one_launch_bit_for_bit as _check

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import gpu_util
    return gpu_util


# (Cin, Ce, Cout, stride, residual) per block
CHAINS = {
    "odd_maps": (7, [(8, 48, 8, 1, True), (8, 40, 24, 2, False), (24, 144, 24, 1, True), (24, 144, 40, 2, False), (40, 240, 40, 1, True)]),
    "one_to_one": (3, [(56, 336, 56, 1, True), (56, 336, 72, 2, False), (72, 100, 72, 1, True)]),
    "large_first": (24, [(8, 48, 8, 2, False), (8, 48, 8, 1, True), (8, 48, 24, 2, False)]),
    "wide": (3, [(32, 192, 56, 1, False), (56, 336, 56, 1, True), (56, 336, 112, 1, False), (112, 320, 128, 1, False)]),  # late weights
}


@pytest.mark.parametrize("N", [1, 3, 300])
@pytest.mark.parametrize("name", list(CHAINS))
def test_image_chain_bit_for_bit(G, name, N):
    H, blocks = CHAINS[name]
    _check(G, N, H, blocks)


def test_chain_of_more_images_than_that_bit_for_bit(G):
    """Past two images a CU the chain of tiles of several images runs."""
    _check(G, 700, 6, [(24, 144, 24, 1, True), (24, 144, 32, 1, False), (32, 192, 32, 1, True)])
