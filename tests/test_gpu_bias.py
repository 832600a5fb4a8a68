"""The bias of the layer: added in the epilogue of the GEMM of a forward, whichever kernel that is, by a kernel of its own behind the
GEMMs of a whole step on more than 256 tokens and output features, and its gradient as column sums."""
import pytest
import torch

from conftest import make_gen, randn_bf16

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def T():
    import triton_int8_amd
    return triton_int8_amd


# few rows, medium, 256 x 128 tiles (odd number of K tiles), 256 x 256 tiles, rows behind the last token; both accumulations
@pytest.mark.parametrize("scheme,had", [("block_channel", None), ("row_block", 128), ("double_channel", None)])
@pytest.mark.parametrize("tokens,k,n", [(1, 512, 384), (33, 1024, 512), (256, 512, 1024), (300, 512, 384), (1000, 1024, 1152), (4100, 1152, 4096), (8192, 512, 4096)])
def test_bias_is_the_rounded_sum(T, dev, scheme, had, tokens, k, n):
    g = make_gen(tokens + n)
    x, b = randn_bf16(g, tokens, k).to(dev), randn_bf16(g, n, std=3.0).to(dev)
    b[:2] = torch.tensor([float("inf"), float("nan")], device=dev)
    lin = T.Int8Linear(k, n, bias=True, scheme=scheme, hadamard=had, device=dev)
    with torch.no_grad():
        plain = lin(x)              # the bias is zero: Y itself (-0 aside, which compares equal)
        lin.bias.copy_(b)
        want = plain + b
        assert torch.equal(torch.nan_to_num(lin(x)), torch.nan_to_num(want))
    assert torch.equal(torch.nan_to_num(lin(x).detach()), torch.nan_to_num(want))
    # a bias that the kernels do not take (not 16-byte aligned) is added by torch
    shifted = torch.empty(n + 1, dtype=torch.bfloat16, device=dev)[1:]
    shifted.copy_(b)
    lin.bias = torch.nn.Parameter(shifted)
    with torch.no_grad():
        assert torch.equal(torch.nan_to_num(lin(x)), torch.nan_to_num(want))


# what is left of the tilings: 128 x 128 on four waves, a round of 256 x 128; rows of scales on both operands and on neither
@pytest.mark.parametrize("scheme,had", [("block_channel", None), ("block_channel", 128), ("row_block", None), ("double_channel", None)])
@pytest.mark.parametrize("tokens,k,n", [(1400, 384, 3072), (2048, 256, 4096), (5000, 256, 2176)])
def test_bias_in_the_epilogue_of_large_tiles(T, dev, scheme, had, tokens, k, n):
    g = make_gen(tokens + n)
    x, w, b = randn_bf16(g, tokens, k).to(dev), randn_bf16(g, n, k).to(dev), randn_bf16(g, n, std=30.0).to(dev)
    call = lambda bias: T.ops.linear_call(T._lib.PART_FORWARD, scheme, had, tokens, k, n, X=x, W=w, bias=bias)[0][:tokens]
    assert torch.equal(call(b), call(None) + b)


# forward and backward in one call: Y beside dX and dW in one launch or two (few tokens), with a launch of its own (few output features), and
# behind the GEMMs by the kernel that adds a bias
@pytest.mark.parametrize("scheme", ["block_channel", "row_block", "double_channel"])
@pytest.mark.parametrize("tokens,k,n", [(16, 512, 640), (16, 1152, 256), (200, 2048, 4096), (300, 512, 256), (1000, 384, 1152)])
def test_bias_of_a_whole_step(T, dev, scheme, tokens, k, n):
    g = make_gen(tokens + n)
    x, w, dy, b = (t.to(dev) for t in (randn_bf16(g, tokens, k), randn_bf16(g, n, k), randn_bf16(g, tokens, n), randn_bf16(g, n, std=30.0)))
    both = T._lib.PART_FORWARD | T._lib.PART_BACKWARD
    call = lambda bias: T.ops.linear_call(both, scheme, None, tokens, k, n, X=x, W=w, dY=dy, one_launch=False, bias=bias)
    (y, dx, dw, _), want = call(b), call(None)
    assert torch.equal(y[:tokens], want[0][:tokens] + b)
    assert torch.equal(dx[:tokens], want[1][:tokens]) and torch.equal(dw, want[2])


@pytest.mark.parametrize("rows,cols", [(1, 32), (5, 96), (16, 512), (17, 544), (1500, 5632), (4099, 128), (3000, 14336)])
def test_column_sum(T, dev, rows, cols):
    g = make_gen(rows + cols)
    wide = randn_bf16(g, rows, cols + 8).to(dev)
    for x in (wide[:, :cols].contiguous(), wide[:, :cols]):     # dense, and rows with a gap
        exact = x.double().sum(0)
        got = T.ops.column_sum(x)
        # one rounding to bf16 (2^-9) and at most log2-ish chains of fp32 additions, each 2^-24 of the sum of magnitudes
        bound = exact.abs() * 2.0 ** -8 + x.double().abs().sum(0) * (rows / 4 + 16) * 2.0 ** -24
        assert bool(((got.double() - exact).abs() <= bound).all())
    assert T.ops.column_sum(torch.full((rows, cols), float("inf"), dtype=torch.bfloat16, device=dev)).isinf().all()


# the last rows and columns that one launch takes, and the first that two take
@pytest.mark.parametrize("rows,cols", [(255, 8192), (3072, 1056), (3073, 1056), (1024, 8224), (1025, 8224)])
def test_column_sum_in_one_launch_and_in_two(T, dev, rows, cols):
    test_column_sum(T, dev, rows, cols)


def test_bias_gradient_can_be_differentiated_again(T, dev):
    lin = T.Int8Linear(256, 128, bias=True, device=dev)
    x, dy = torch.randn(5, 256, device=dev).bfloat16(), torch.ones(5, 128, device=dev).bfloat16().requires_grad_(True)
    (db,) = torch.autograd.grad(lin(x), lin.bias, dy, create_graph=True)
    (back,) = torch.autograd.grad(db.sum(), dy)
    assert torch.equal(back, torch.ones_like(back))
