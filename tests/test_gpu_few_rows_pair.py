"""Y and dX of a step on few tokens as one launch of the few-rows kernel, against the GEMMs launched one by one."""
import pytest
import torch

from conftest import make_gen, randn_bf16

pytestmark = pytest.mark.gpu


# one block row and eight; strips that are and are not a multiple of 8; Y and dX of very different size; one of the two on another kernel
@pytest.mark.parametrize("scheme", ["block_channel", "row_block", "double_channel"])
@pytest.mark.parametrize("tokens,k,n", [(1, 128, 128), (16, 4096, 384), (33, 384, 2048), (128, 1152, 640), (256, 512, 512), (200, 1024, 4096)])
def test_step_on_few_tokens(dev, tokens, k, n, scheme):
    import triton_int8_amd as T
    from triton_int8_amd._lib import PART_BACKWARD, PART_FORWARD, PART_KEEP
    g = make_gen(tokens + k + n)
    X, W, dY = randn_bf16(g, tokens, k).to(dev), randn_bf16(g, n, k, std=0.02).to(dev), randn_bf16(g, tokens, n, std=1e-3).to(dev)
    Y, dX, dW = T.linear_fwd_bwd(X, W, dY, scheme)
    Y1, _, _, saved = T.ops.linear_call(PART_FORWARD | PART_KEEP, scheme, None, tokens, k, n, X=X, W=W)
    _, dX1, dW1, _ = T.ops.linear_call(PART_BACKWARD | PART_KEEP, scheme, None, tokens, k, n, X=X, W=W, dY=dY, saved=saved)
    assert torch.equal(Y, Y1[:tokens]) and torch.equal(dX, dX1[:tokens]) and torch.equal(dW, dW1)
