"""Up to 8 rows through a quantised weight: the kernel that quantises them itself gives the bits of quantiser and GEMM apart."""
import pytest
import torch

import triton_int8_amd as T
from triton_int8_amd._lib import PART_FORWARD

pytestmark = pytest.mark.gpu


# one to eight rows (nine: quantiser and GEMM apart); one K tile (three waves without one), as many as waves, a ragged split, more than 64,
# too many on few columns (apart) and on many; a single strip of columns group and strips that share an XCD
@pytest.mark.parametrize("tokens", [1, 3, 7, 8])
@pytest.mark.parametrize("k, n", [(128, 128), (512, 384), (1152, 1024), (9088, 256), (10368, 128), (14336, 128), (32768, 8320)])
@pytest.mark.parametrize("scheme, bias", [("block_channel", False), ("block_channel", True), ("row_block", True), ("double_channel", True)])
def test_bits(dev, tokens, k, n, scheme, bias):
    g = torch.Generator(device=dev).manual_seed(tokens * k + n)
    wide = torch.randn(9, k + 8, generator=g, device=dev)
    wide[:, ::101] *= 30.0
    wide[:, 128:256] = 0.0 if k > 256 else 1.0      # a K tile of zeros, a row of zeros: the floor of the absmax
    if tokens > 2:
        wide[1] = 0.0
    wide = wide.to(torch.bfloat16)
    wide[tokens:] = 0.0                             # further rows of zeros leave the others' scales as they are
    W = torch.randn(n, k, generator=g, device=dev).to(torch.bfloat16)
    b = torch.randn(n, generator=g, device=dev).to(torch.bfloat16) if bias else None
    wq = T.linear.quantize_weight(W, scheme, None)
    call = lambda x: T.ops.linear_call(PART_FORWARD, scheme, None, x.shape[0], k, n, X=x, wq=wq, bias=b)[0][:tokens]
    apart = call(wide[:9, :k])
    assert torch.equal(call(wide[:tokens, :k]), apart) and torch.equal(call(wide[:tokens, :k].contiguous()), apart)
    # what is not finite goes the same way
    wide[0, 5], wide[0, k // 2] = float("nan"), float("inf")
    assert torch.equal(call(wide[:tokens, :k]).view(torch.int16), call(wide[:9, :k]).view(torch.int16))
