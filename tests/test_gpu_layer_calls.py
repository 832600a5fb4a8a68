"""The layer calls queued from C (ti8_linear, ti8_linear_quantise, ti8_linear_fwd_bwd) on any number of tokens against the
step assembled from the separate entry points on zero-padded copies: the same bits, whatever lies in memory behind the last
token."""
import pytest
import torch

from conftest import make_gen, randn_bf16

pytestmark = pytest.mark.gpu

MODES = [("block_channel", None), ("row_block", None), ("double_channel", None), ("block_channel", 128), ("row_block", 128), ("double_channel", "full")]


@pytest.fixture(scope="module")
def T():
    import triton_int8_amd
    return triton_int8_amd


def tokens_in_a_bigger_buffer(g, dev, tokens, cols, std=1.0):
    """[tokens, cols] whose buffer goes on with NaN: a kernel that reads past the last token shows it."""
    buf = torch.full((tokens + 128, cols), float("nan"), dtype=torch.bfloat16, device=dev)
    buf[:tokens] = randn_bf16(g, tokens, cols, std=std).to(dev)
    return buf[:tokens]


@pytest.mark.parametrize("tokens", [1, 33, 127, 128, 129, 300, 641])
@pytest.mark.parametrize("scheme,had", MODES)
def test_layer_calls_match_the_assembled_step(T, dev, monkeypatch, scheme, had, tokens):
    g = make_gen(tokens * 7 + len(scheme))
    K, N = 512, 384 if had != "full" else 512
    X, dY = tokens_in_a_bigger_buffer(g, dev, tokens, K), tokens_in_a_bigger_buffer(g, dev, tokens, N, 1e-3)
    W = randn_bf16(g, N, K, std=0.02).to(dev)
    step = T.linear_fwd_bwd(X, W, dY, scheme, had)
    lin = T.Int8Linear(K, N, bias=True, scheme=scheme, hadamard=had, device=dev)
    with torch.no_grad():
        lin.weight.copy_(W)
        lin.bias.copy_(randn_bf16(g, N).to(dev))

    def module():
        x = X.clone().requires_grad_(True)
        y = lin(x)
        grads = torch.autograd.grad(y, (x, lin.weight, lin.bias), dY)
        with torch.no_grad():
            return [y.detach(), *grads, lin(X)]
    from_c = module()
    monkeypatch.setattr(T.linear, "ONE_CALL_STEP", False)
    for name, got, want in zip(("Y", "dX", "dW"), step, T.linear_fwd_bwd(X, W, dY, scheme, had)):
        assert got.shape == want.shape and torch.isfinite(got).all() and torch.equal(got, want), name
    for name, got, want in zip(("y", "dx", "dw", "db", "y without autograd"), from_c, module()):
        assert got.shape == want.shape and torch.isfinite(got).all() and torch.equal(got, want), name


@pytest.mark.parametrize("scheme,had", MODES)
def test_backward_without_what_the_forward_kept(T, dev, scheme, had):
    """ti8_linear with TI8_PART_BACKWARD alone quantises X and W again: the bits of the backward that reuses them."""
    from triton_int8_amd._lib import PART_BACKWARD, PART_FORWARD, PART_KEEP
    g = make_gen(17)
    K, N, tokens = 512, 512, 300
    X, dY, W = tokens_in_a_bigger_buffer(g, dev, tokens, K), tokens_in_a_bigger_buffer(g, dev, tokens, N, 1e-3), randn_bf16(g, N, K, std=0.02).to(dev)
    Y, _, _, saved = T.ops.linear_call(PART_FORWARD | PART_KEEP, scheme, had, tokens, K, N, X=X, W=W)
    _, dX, dW, _ = T.ops.linear_call(PART_BACKWARD | (PART_KEEP if saved is not None else 0), scheme, had, tokens, K, N, X=X, W=W, dY=dY, saved=saved)
    _, dX2, dW2, _ = T.ops.linear_call(PART_BACKWARD, scheme, had, tokens, K, N, X=X, W=W, dY=dY, one_launch=False)
    assert torch.equal(dX[:tokens], dX2[:tokens]) and torch.equal(dW, dW2)
    assert (saved is None) == (had is not None)


def test_layer_call_validation(T, dev):
    from triton_int8_amd._lib import PART_BACKWARD, PART_FORWARD
    X, W = torch.zeros(5, 256, dtype=torch.bfloat16, device=dev), torch.zeros(128, 256, dtype=torch.bfloat16, device=dev)
    with pytest.raises(ValueError, match="do not fit"):
        T.linear_fwd_bwd(X, W, torch.zeros(4, 128, dtype=torch.bfloat16, device=dev), "row_block")
    with pytest.raises(ValueError, match="multiples of 128"):
        T.ops.linear_call(PART_FORWARD, "row_block", None, 5, 200, 128, X=X, W=W)
    with pytest.raises(T._lib.Ti8Error, match="required"):
        T.ops.linear_call(PART_BACKWARD, "row_block", None, 5, 256, 128, X=X, W=W, one_launch=False)
    with pytest.raises(ValueError, match="bfloat16"):
        T.ops.linear_call(PART_FORWARD, "row_block", None, 5, 256, 128, X=X.float(), W=W)
