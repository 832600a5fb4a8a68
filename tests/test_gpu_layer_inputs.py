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
