"""GEMMs over different numbers of K tiles in one launch of persistent workgroups, which take their tiles from lists: the bits of one
workgroup per tile, over NaN-filled outputs."""
import pytest
import torch

import triton_int8_amd as T
from triton_int8_amd._lib import KERNEL_PERSISTENT_CHAIN, SCALE_BLOCK128, SCALE_ROW

pytestmark = pytest.mark.gpu


# the three GEMMs of a step and the two of its backward: fewer tiles than workgroups in all, the longest in a part of them; several rounds, numbers
# of tiles that 8 does not divide, tiles that hang over; an odd number of K tiles among them (13, 27); a list of more rounds than GEMMs
@pytest.mark.parametrize("tokens, k, n", [(512, 8192, 1024), (1280, 9216, 2688), (1664, 6912, 5760), (3456, 1280, 6656), (2304, 10752, 1536)])
@pytest.mark.parametrize("first", [0, 1])
@pytest.mark.parametrize("row_block", [False, True])
def test_bits(dev, monkeypatch, tokens, k, n, first, row_block):
    from triton_int8_amd import ops
    g = torch.Generator(device=dev).manual_seed(tokens + k + n)

    def operand(rows, cols, mode):
        q = torch.randint(-127, 128, (rows, cols), generator=g, dtype=torch.int8, device=dev)
        return q, torch.rand(*((rows,) if mode == SCALE_ROW else (rows // 128, cols // 128)), generator=g, device=dev) + 0.5

    modes = [(SCALE_ROW, SCALE_BLOCK128)] * 3 if row_block else [(SCALE_BLOCK128, SCALE_ROW)] * 2 + [(SCALE_BLOCK128, SCALE_BLOCK128)]
    problems = []
    for (M, N, K), (mA, mB) in list(zip(((tokens, n, k), (tokens, k, n), (n, k, tokens)), modes))[first:]:
        (A, sA), (B, sB) = operand(M, K, mA), operand(N, K, mB)
        problems.append(dict(A=A, B=B, sA=sA, modeA=mA, sB=sB, modeB=mB))
    monkeypatch.setattr(ops, "GEMM_PATH", "large")
    results = []
    for persistent in (True, False):
        monkeypatch.setattr(ops, "GEMM_PERSISTENT", persistent)
        for p in problems:
            p["out"] = torch.full((p["A"].shape[0], p["B"].shape[0]), float("nan"), dtype=torch.bfloat16, device=dev)
        results.append(ops.gemm_i8_nt_multi(problems, together=True))
        assert (T.last_gemm_kernel() == KERNEL_PERSISTENT_CHAIN) == persistent
    for got, want in zip(*results):
        assert torch.equal(got, want) and torch.isfinite(got).all()
