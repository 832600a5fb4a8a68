"""GEMMs over different numbers of K tiles in one launch of persistent workgroups, which take their tiles from lists: the bits of one
workgroup per tile, over NaN-filled outputs."""
import pytest
import torch

import triton_int8_amd as T
from triton_int8_amd._lib import FORM_LISTS, FORM_PLAIN, KERNEL_PERSISTENT_CHAIN, SCALE_BLOCK128, SCALE_ROW, last_gemm_form

pytestmark = pytest.mark.gpu


# the three GEMMs of a step and the two of its backward, and whether they come from lists on 256 CUs: by rounds where a workgroup has one tile at
# most or rounds are as good; two GEMMs and three, several rounds, numbers of tiles that 8 does not divide, tiles that hang over; an odd
# number of K tiles among them (13, 17, 27, 29, 51); nearly as many entries as a list has
@pytest.mark.parametrize("tokens, k, n, first, lists", [
    (512, 8192, 1024, 0, False), (1280, 9216, 2688, 0, True), (1664, 6912, 5760, 0, True), (3456, 1280, 6656, 0, True), (2304, 10752, 1536, 0, True),
    (512, 8192, 1024, 1, False), (1280, 9216, 2688, 1, False), (1664, 6912, 5760, 1, False), (3456, 1280, 6656, 1, False), (2304, 10752, 1536, 1, False),
    (1536, 4736, 3712, 1, True), (3456, 4992, 1536, 1, True), (2176, 2944, 6528, 1, True), (1536, 14336, 14336, 0, True)])
@pytest.mark.parametrize("row_block", [False, True])
def test_bits(dev, monkeypatch, tokens, k, n, first, lists, row_block):
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
        assert (T.last_gemm_kernel() == KERNEL_PERSISTENT_CHAIN) == persistent and last_gemm_form() == (FORM_LISTS if persistent and lists else FORM_PLAIN)
    for got, want in zip(*results):
        assert torch.equal(got, want) and torch.isfinite(got).all()
