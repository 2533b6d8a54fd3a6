"""Outputs of 24 to 256 MB are stored through the L2 so that they stay in the last-level cache, others past it: every element of outputs on
either side of both limits is written, tails included, by each operator's vector width."""
import numpy as np
import pytest
import torch

from oracle import oracle as zo

pytestmark = pytest.mark.gpu

MB = 1 << 20


@pytest.fixture(scope="module")
def G():
    import gpu_util
    return gpu_util


# bytes of the output: below and above the lower limit, with and without a tail, above the upper one
@pytest.mark.parametrize("nbytes", [24 * MB - 12, 24 * MB + 4, 24 * MB + 4096, 256 * MB + 20])
def test_f32_operators_write_all_of_their_outputs(G, nbytes):
    n = nbytes // 4
    x = torch.randn(n, device="cuda", generator=torch.Generator("cuda").manual_seed(n))
    y = torch.full_like(x, 7.0)
    v = (1, 1, 1, n)
    G.tm.leakyReLU_lean(x.view(v), 0.1, y.view(v))
    assert torch.equal(y, torch.where(x <= 0, 0.1 * x, x))
    G.tm.sum_tensors_lean(x, y, y2 := torch.full_like(x, 7.0))
    assert torch.equal(y2, x + y)
    q = torch.randint(0, 256, (n,), device="cuda", dtype=torch.uint8)
    s, z = torch.tensor([0.03], device="cuda"), torch.tensor([120], dtype=torch.uint8, device="cuda")
    G.tm.dequantize_linear(q, s, z, 0, out=y)
    assert torch.equal(y, (q.int() - 120).float() * s)


@pytest.mark.parametrize("n", [24 * MB - 3, 24 * MB + 5, 24 * MB + 16])
def test_u8_operators_write_all_of_their_outputs(G, n):
    g = torch.Generator("cuda").manual_seed(n)
    x = torch.randn(n, device="cuda", generator=g)
    s, z = torch.tensor([0.03], device="cuda"), torch.tensor([120], dtype=torch.uint8, device="cuda")
    q = torch.full((n,), 9, dtype=torch.uint8, device="cuda")
    G.tm.quantize_linear(x, s, z, 0, out=q)
    assert torch.equal(q, ((x / s).round() + 120).clamp(0, 255).to(torch.uint8))
    a = torch.full_like(q, 9)
    G.tm.qlinear_act(q, 0.03, 120, "relu", 0.0, 0.03, 120, out=a)
    assert torch.equal(a, q.clamp(min=120))
    b = torch.full_like(q, 9)
    G.tm.qlinear_add(q, 0.5, 120, a, 0.5, 120, 0.5, 120, out=b)
    assert torch.equal(b, (q.int() + a.int() - 120).clamp(0, 255).to(torch.uint8))


@pytest.mark.parametrize("planes", [9000, 9477])
def test_plane_operators_write_all_of_their_outputs(G, planes):
    """26x26 and 27x27 planes on both sides of the lower limit: normalisation, pools, resize, concatenation."""
    for H in (26, 27):
        x = torch.randn(planes, 1, H, H, device="cuda", generator=torch.Generator("cuda").manual_seed(planes + H))
        one, zero = torch.ones(1, device="cuda"), torch.zeros(1, device="cuda")
        y = torch.full_like(x, 7.0)
        G.tm.batchnorm(x, 2 * one, one, zero, one, 0.0, out=y)
        assert torch.equal(y, x / one * 2 + 1)
        big = x.view(1, planes, H, H).expand(5, planes, H, H).contiguous()
        for pool in (torch.nn.functional.max_pool2d, torch.nn.functional.avg_pool2d):
            p = torch.full((5, planes, H // 2, H // 2), 7.0, device="cuda")
            if pool is torch.nn.functional.max_pool2d:
                G.tm.onnx_maxpool_lean(big, p, [2, 2], [2, 2], [1, 1], [0, 0, 0, 0])
                assert torch.equal(p, pool(big, 2))
            else:
                G.tm.avgpool_lean(big, p, [2, 2], [2, 2])
                # four values, each partial sum rounded once
                assert ((p - pool(big, 2)).abs() <= 2.0 ** -22 * pool(big.abs(), 2)).all()
        half = x[:, :, :13, :13].contiguous()
        r = torch.full((planes, 1, 26, 26), 7.0, device="cuda")
        G.tm.resize(half, "nearest", None, list(r.shape), "asymmetric", out=r)
        assert (r.cpu().numpy() == zo.resize(half.cpu().numpy(), "nearest", None, list(r.shape), "asymmetric")).all()
        c = torch.full((planes, 2, H, H), 7.0, device="cuda")
        G.tm.lean_concatenate([x, y], 1, c)
        assert torch.equal(c, torch.cat([x, y], 1))


@pytest.mark.parametrize("H", [48, 24, 26, 27])
def test_u8_pools_write_all_of_their_outputs(G, H):
    """Rows of whole vectors, whole planes in LDS, and rows at any alignment, just below and above the lower limit."""
    per = (H // 2) ** 2
    for planes in (24 * MB // per, 24 * MB // per + 3):
        x = torch.randint(0, 256, (1, planes, H, H), device="cuda", dtype=torch.uint8, generator=torch.Generator("cuda").manual_seed(planes))
        y = torch.full((1, planes, H // 2, H // 2), 9, dtype=torch.uint8, device="cuda")
        G.tm.onnx_maxpool_lean(x, y, [2, 2], [2, 2], [1, 1], [0, 0, 0, 0])
        v = x[:, :, :H // 2 * 2, :H // 2 * 2].reshape(1, planes, H // 2, 2, H // 2, 2)
        assert torch.equal(y, v.amax((3, 5)))


@pytest.mark.parametrize("rows", [24 * MB // 40 - 3, 24 * MB // 40 + 1, 24 * MB // 40 + 259])
def test_softmax_of_short_rows_writes_all_of_its_output(G, rows):
    x = torch.randn(rows, 10, device="cuda", generator=torch.Generator("cuda").manual_seed(rows))
    y = torch.full_like(x, 7.0)
    G.tm.softmax_lean(x, y)
    want = torch.softmax(x.double(), 1)
    # an exponential and nine additions of at most half a unit in the last place each, a division: 16 units of 2^-24 at the most
    assert ((y - want).abs() <= 16 * 2.0 ** -24 * want).all()


@pytest.mark.parametrize("planes", [9300, 9310])
def test_a_term_a_channel_is_added_to_all_of_the_output(G, planes):
    x = torch.randn(5, planes // 5, 26, 26, device="cuda", generator=torch.Generator("cuda").manual_seed(planes))
    c = torch.randn(1, planes // 5, 1, 1, device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    y = torch.full_like(x, 7.0)
    G.tm.sum_tensors_lean(x, c, y)
    assert torch.equal(y, x + c)


@pytest.mark.parametrize("side", [26, 27, 32])
def test_u8_resize_and_concatenation_write_all_of_their_outputs(G, side):
    """Outputs just above the lower limit; pieces of whole 16 bytes, of four and of single ones."""
    n = 24 * MB // (2 * side * side) + 2
    x = torch.randint(0, 256, (n, 1, side, side), device="cuda", dtype=torch.uint8, generator=torch.Generator("cuda").manual_seed(side))
    c = torch.full((n, 2, side, side), 9, dtype=torch.uint8, device="cuda")
    G.tm.lean_concatenate([x, 255 - x], 1, c)
    assert torch.equal(c, torch.cat([x, 255 - x], 1))
    small = x.repeat(2, 1, 1, 1)[:, :, :13, :13].contiguous()
    r = torch.full((2 * n, 1, side, side), 9, dtype=torch.uint8, device="cuda")
    G.tm.resize(small, "nearest", None, list(r.shape), "asymmetric", out=r)
    # the oracle's rule for rows and columns, from one map of their numbers
    number = np.broadcast_to(np.arange(13, dtype=np.uint8), (1, 1, 13, 13))
    at = torch.from_numpy(zo.resize(np.ascontiguousarray(number), "nearest", None, [1, 1, side, side], "asymmetric")[0, 0, 0].astype(np.int64)).cuda()
    assert torch.equal(r, small[:, :, at][:, :, :, at])
