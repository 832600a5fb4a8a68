"""Up to 8 rows on few columns: 16 columns per workgroup, codes of 8 K tiles at a time, give the bits of quantiser and GEMM apart."""
import pytest
import torch

import triton_int8_amd as T
from triton_int8_amd._lib import FORM_ROWS_NARROW, PART_FORWARD, last_gemm_form

pytestmark = pytest.mark.gpu


# every instance by rows (1, 2, 4, 8) full and not; a wave without a K tile, one batch of 8 not full, full, one K tile more, and several
# (up to 4 rows these go to it at any K, 5 to 8 from 24 K tiles on); one workgroup per CU, and one strip more, which goes elsewhere
@pytest.mark.parametrize("tokens", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("k, n", [(256, 128), (3072, 128), (4096, 384), (4224, 256), (11776, 128), (4096, 4096), (4096, 4224)])
@pytest.mark.parametrize("scheme, bias", [("block_channel", True), ("row_block", False), ("double_channel", False), ("double_channel", True)])
def test_bits(dev, tokens, k, n, scheme, bias):
    g = torch.Generator(device=dev).manual_seed(100 * tokens + k + n)
    wide = torch.randn(9, k + 8, generator=g, device=dev)
    wide[:, ::101] *= 30.0
    wide[:, 128:256] = 0.0                          # a K tile of zeros and a row of zeros: the floor of the absmax
    if tokens > 2:
        wide[1] = 0.0
    wide = wide.to(torch.bfloat16)
    wide[tokens:] = 0.0                             # further rows of zeros leave the others' scales as they are
    W = torch.randn(n, k, generator=g, device=dev).to(torch.bfloat16)
    b = torch.randn(n, generator=g, device=dev).to(torch.bfloat16) if bias else None
    wq = T.linear.quantize_weight(W, scheme, None)
    call = lambda x: T.ops.linear_call(PART_FORWARD, scheme, None, x.shape[0], k, n, X=x, wq=wq, bias=b)[0][:tokens]
    apart = call(wide[:9, :k])
    assert last_gemm_form() != FORM_ROWS_NARROW
    assert torch.equal(call(wide[:tokens, :k]), apart) and torch.equal(call(wide[:tokens, :k].contiguous()), apart)
    assert (last_gemm_form() == FORM_ROWS_NARROW) == (n <= 4096 and (tokens <= 4 or k >= 3072))
    wide[0, 5], wide[0, k // 2] = float("nan"), float("inf")
    assert torch.equal(call(wide[:tokens, :k]).view(torch.int16), call(wide[:9, :k]).view(torch.int16))
