"""The persistent kernel on an odd number of K tiles, walked as one more: the bits of one workgroup per tile."""
import pytest
import torch

import triton_int8_amd as T
from triton_int8_amd._lib import COMBINE_DIV_PROD, COMBINE_MUL_MUL, KERNEL_ONE_TILE, KERNEL_PERSISTENT_CHAIN, SCALE_BLOCK128, SCALE_ROW

pytestmark = pytest.mark.gpu


# the fewest that go there and one less; one before, at and behind a refill of the factors; the most; one tile per workgroup and several, tiles
# that hang over; the largest scale on the last K tile, which would show if it counted twice
@pytest.mark.parametrize("nk", [17, 19, 21, 63, 65, 127, 129, 255])
@pytest.mark.parametrize("M, N", [(384, 640), (4224, 4352)])
@pytest.mark.parametrize("modes, combine", [((SCALE_BLOCK128, SCALE_ROW), COMBINE_MUL_MUL), ((SCALE_ROW, SCALE_BLOCK128), COMBINE_MUL_MUL),
                                            ((SCALE_BLOCK128, SCALE_BLOCK128), COMBINE_DIV_PROD)])
def test_bits(dev, monkeypatch, nk, M, N, modes, combine):
    from triton_int8_amd import ops
    if nk > 65 and M > 384:
        M, N = 2176, 2304
    g = torch.Generator(device=dev).manual_seed(nk * M)
    K = 128 * nk
    A, B = (torch.randint(-127, 128, s, generator=g, dtype=torch.int8, device=dev) for s in ((1, M, K), (N, K)))

    def scale(rows, mode, batch):
        s = torch.rand(*((rows,) if mode == SCALE_ROW else (rows // 128, nk)), generator=g, device=dev) + 0.25
        if mode != SCALE_ROW:
            s[:, -1] *= 5.0
        return s[None] if batch else s

    sA, sB = scale(M, modes[0], True), scale(N, modes[1], False)
    monkeypatch.setattr(ops, "GEMM_PATH", "large")
    outs = []
    for persistent in (True, False):
        monkeypatch.setattr(ops, "GEMM_PERSISTENT", persistent)
        outs.append(torch.full((1, M, N), float("nan"), dtype=torch.bfloat16, device=dev))
        ops.gemm_i8_nt(A, B, sA, modes[0], sB, modes[1], combine=combine, out=outs[-1])
        assert T.last_gemm_kernel() == (KERNEL_PERSISTENT_CHAIN if persistent and nk >= 19 else KERNEL_ONE_TILE)
    assert torch.equal(*outs) and torch.isfinite(outs[0]).all()
