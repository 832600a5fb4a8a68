"""Inputs of the layer that are not plain dense tensors: gradients and activations broadcast over the rows, tensors at odd offsets,
biases of another type or with a gradient of their own, very many tokens."""
import pytest
import torch

from conftest import make_gen, randn_bf16

pytestmark = pytest.mark.gpu

MODES = [("block_channel", None), ("row_block", None), ("double_channel", None), ("block_channel", 128), ("row_block", 128), ("double_channel", "full")]
K, N = 512, 512


@pytest.fixture(scope="module")
def T():
    import triton_int8_amd
    return triton_int8_amd


def layer(T, g, dev, scheme, had, bias=True):
    lin = T.Int8Linear(K, N, bias=bias, scheme=scheme, hadamard=had, device=dev)
    with torch.no_grad():
        lin.weight.copy_(randn_bf16(g, N, K, std=0.02))
        if bias:
            lin.bias.copy_(randn_bf16(g, N))
    return lin


# a bias that the kernels add, and one that torch adds (not 16-byte aligned)
@pytest.mark.parametrize("aligned", [True, False])
@pytest.mark.parametrize("tokens", [5, 300, 1024])
@pytest.mark.parametrize("scheme,had", MODES)
def test_bias_gradient_behind_a_frozen_weight(T, dev, scheme, had, tokens, aligned):
    g = make_gen(tokens)
    lin = layer(T, g, dev, scheme, had)
    if not aligned:
        lin.bias = torch.nn.Parameter(torch.cat((lin.bias[:1], lin.bias))[1:].detach())
        assert lin.bias.data_ptr() % 16
    lin.weight.requires_grad_(False)
    x, dy = randn_bf16(g, tokens, K).to(dev), randn_bf16(g, tokens, N).to(dev)
    y = lin(x)
    assert y.requires_grad
    (db,) = torch.autograd.grad(y, lin.bias, dy)
    assert torch.equal(db, dy.sum(0))
    with torch.no_grad():
        assert torch.equal(y, lin(x)) and not lin(x).requires_grad
    assert not lin.requires_grad_(False)(x).requires_grad


def step_and_module(T, lin, scheme, had, x, dy, backward):
    """What the entry points return for the tensors as they are: the one-call step, the module without autograd and with it."""
    bias, lin.bias = lin.bias, None
    with torch.no_grad():
        outs = [*T.linear_fwd_bwd(x, lin.weight.detach(), dy, scheme, had), lin(x)]
    lin.bias = bias
    leaf = x.detach().requires_grad_(True)
    assert leaf.stride() == x.stride() and leaf.data_ptr() == x.data_ptr()
    y = lin(leaf)
    return [*outs, y.detach(), *backward(y, (leaf, lin.weight, lin.bias))]


def compare_with_dense(T, dev, scheme, had, lin, x, dy, backward):
    dense = [torch.empty(t.shape, dtype=t.dtype, device=dev).copy_(t) for t in (x, dy)]
    want = step_and_module(T, lin, scheme, had, *dense, lambda y, leaves: torch.autograd.grad(y, leaves, dense[1]))
    got = step_and_module(T, lin, scheme, had, x, dy, backward)
    for name, a, b in zip(("Y", "dX", "dW", "y without autograd", "y", "dx", "dw", "db"), got, want):
        assert torch.isfinite(a).all() and torch.equal(a, b), name


@pytest.mark.parametrize("tokens", [1, 5, 128, 300, 512])
@pytest.mark.parametrize("scheme,had", MODES)
def test_rows_broadcast_from_one(T, dev, scheme, had, tokens):
    """One row for all tokens: the gradient that a sum over the tokens sends back, and an activation expanded over a batch."""
    g = make_gen(tokens)
    lin = layer(T, g, dev, scheme, had)
    row_x, row_dy = randn_bf16(g, 7, K).to(dev), randn_bf16(g, N, std=1e-3).to(dev)
    x, dy = row_x[3:4].expand(8 * tokens, K)[:tokens], row_dy.expand(8 * tokens, N)[:tokens]
    assert x.stride(0) == dy.stride(0) == 0
    compare_with_dense(T, dev, scheme, had, lin, x, dy, lambda y, leaves: torch.autograd.grad(y.sum(0), leaves, row_dy))


@pytest.mark.parametrize("tokens", [1, 300, 512])
@pytest.mark.parametrize("scheme,had", MODES)
def test_rows_that_overlap(T, dev, scheme, had, tokens):
    g = make_gen(tokens)
    lin = layer(T, g, dev, scheme, had)
    x, dy = randn_bf16(g, 8 * tokens + K).to(dev).as_strided((tokens, K), (8, 1)), randn_bf16(g, 8 * tokens + N, std=1e-3).to(dev).as_strided((tokens, N), (8, 1))
    compare_with_dense(T, dev, scheme, had, lin, x, dy, lambda y, leaves: torch.autograd.grad(y, leaves, dy))


@pytest.mark.parametrize("tokens", [1, 5, 128, 300])
@pytest.mark.parametrize("scheme,had", MODES)
def test_rows_at_odd_offsets(T, dev, scheme, had, tokens):
    """Dense tensors that do not start on 16 bytes, and a single row out of rows whose distance is no multiple of 16 bytes."""
    g = make_gen(tokens)
    lin = layer(T, g, dev, scheme, had)
    x, dy = randn_bf16(g, tokens * K + 1).to(dev)[1:].view(tokens, K), randn_bf16(g, tokens * N + 3, std=1e-3).to(dev)[3:].view(tokens, N)
    assert x.is_contiguous() and x.data_ptr() % 16 and dy.is_contiguous() and dy.data_ptr() % 16
    compare_with_dense(T, dev, scheme, had, lin, x, dy, lambda y, leaves: torch.autograd.grad(y, leaves, dy))
    x, dy = randn_bf16(g, tokens, K + 4).to(dev)[:, :K], randn_bf16(g, tokens, N + 4, std=1e-3).to(dev)[:, :N]
    compare_with_dense(T, dev, scheme, had, lin, x, dy, lambda y, leaves: torch.autograd.grad(y, leaves, dy))


@pytest.mark.parametrize("tokens", [5, 300])
@pytest.mark.parametrize("scheme,had", MODES)
def test_bias_of_another_type(T, dev, scheme, had, tokens):
    """A float32 bias: the sum is made and returned in float32, with and without autograd."""
    g = make_gen(tokens)
    lin = layer(T, g, dev, scheme, had, bias=False)
    x, b = randn_bf16(g, tokens, K).to(dev), torch.randn(N, generator=g).to(dev)
    with torch.no_grad():
        want = lin(x) + b
    lin.bias = torch.nn.Parameter(b)
    with torch.no_grad():
        y = lin(x)
        assert y.dtype == torch.float32 and torch.equal(y, want)
    y = lin(x)
    assert y.dtype == torch.float32 and torch.equal(y, want)


def test_a_batch_of_biases(T, dev):
    """vmap over the bias: one GEMM, a sum for each bias."""
    g = make_gen(2)
    lin = layer(T, g, dev, "block_channel", None)
    x, biases = randn_bf16(g, 300, K).to(dev), randn_bf16(g, 3, N).to(dev)
    with torch.no_grad():
        got = torch.func.vmap(lambda b: torch.func.functional_call(lin, {"bias": b}, (x,)))(biases)
        for y, b in zip(got, biases):
            assert torch.equal(y, torch.func.functional_call(lin, {"bias": b}, (x,)))


@pytest.mark.parametrize("scheme", ["row_block", "double_channel"])
def test_more_tokens_than_a_column_pass_takes(T, dev, scheme):
    """Per-row scales: a forward quantises its rows only, and no launch of it has one workgroup row per 32 tokens (at most 65535)."""
    g = make_gen(4)
    tokens, k, n = 65535 * 32 + 129, 128, 128
    lin = T.Int8Linear(k, n, scheme=scheme, device=dev)
    x = torch.randn(tokens, k, generator=torch.Generator(device=dev).manual_seed(4), device=dev, dtype=torch.bfloat16)
    with torch.no_grad():
        y = lin(x)
        for rows in (slice(0, 512), slice(tokens // 2, tokens // 2 + 512), slice(tokens - 512, tokens)):
            assert torch.equal(y[rows], lin(x[rows]))


def test_what_a_column_pass_does_not_take_is_refused(T, dev):
    """The same token counts where an operand is quantised by columns."""
    from triton_int8_amd import ops
    from triton_int8_amd._lib import PART_BACKWARD, PART_FORWARD, PART_KEEP
    tokens, k, n = 65535 * 32 + 1, 128, 128
    big = torch.empty(tokens, k, device=dev, dtype=torch.bfloat16)
    w = torch.empty(n, k, device=dev, dtype=torch.bfloat16)
    for scheme, had, parts in (("row_block", None, PART_BACKWARD), ("row_block", 128, PART_BACKWARD), ("double_channel", None, PART_BACKWARD),
                               ("double_channel", None, PART_FORWARD | PART_KEEP), ("row_block", 128, PART_FORWARD | PART_BACKWARD)):
        with pytest.raises(T._lib.Ti8Error, match="too many tiles"):
            ops.linear_call(parts, scheme, had, tokens, k, n, X=big, W=w, dY=big, one_launch=False)


@pytest.mark.parametrize("scheme,had", MODES)
def test_a_weight_at_the_address_of_the_last(T, dev, scheme, had):
    """Weights that come and go, each likely where the one before it lay: the quantised weight is that of the present one."""
    import copy
    g = make_gen(6)
    lin = layer(T, g, dev, scheme, had, bias=False)
    x = randn_bf16(g, 33, K).to(dev)
    with torch.no_grad():
        for _ in range(3):
            lin(x)
            lin.weight = torch.nn.Parameter(torch.empty(0, dtype=torch.bfloat16, device=dev))
            lin.weight = torch.nn.Parameter(randn_bf16(g, N, K, std=0.02).to(dev))
            fresh = T.Int8Linear(K, N, scheme=scheme, hadamard=had, device=dev)
            fresh.weight.copy_(lin.weight)
            assert torch.equal(lin(x), fresh(x))
        other = copy.deepcopy(lin)
        other.weight.mul_(2.0)
        assert torch.equal(other(x), lin(x) * 2.0) and list(lin.state_dict()) == ["weight"]
