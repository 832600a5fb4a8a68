"""Persistent chained GEMM with operand B scaled per (row, 128 columns), the scales stored column by column, against the one-tile kernel, and the scales' layout."""
import pytest
import torch

from conftest import make_gen, randn_bf16

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def T():
    import triton_int8_amd
    return triton_int8_amd


# (batch, M, N, K): one tile; tiles that hang over M and over N; two K tiles, 64 and 66 (the factor register is refilled); more tiles
# than workgroups; an odd number of K tiles, which the one-tile kernel serves
@pytest.mark.parametrize("batch,M,N,K", [(1, 256, 256, 256), (2, 384, 640, 512), (1, 512, 384, 64 * 128), (1, 256, 512, 66 * 128),
                                         (3, 2304, 2560, 1024), (1, 512, 512, 384)])
def test_lane_scales_on_persistent_workgroups(T, dev, batch, M, N, K):
    from triton_int8_amd._lib import (COMBINE_DIV_PROD, COMBINE_MUL_PROD, KERNEL_ONE_TILE, KERNEL_PERSISTENT_CHAIN, SCALE_BLOCK128,
                                      SCALE_BLOCK_K256, SCALE_ROW, SCALE_ROW_K128)
    ops, g = T.ops, make_gen(M + N + K)
    A = torch.randint(-127, 128, (batch, M, K), generator=g, dtype=torch.int8).to(dev)
    B2 = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8).to(dev)
    B3 = torch.randint(-127, 128, (batch, N, K), generator=g, dtype=torch.int8).to(dev)

    def scale(*shape):
        return torch.rand(shape, generator=g).add_(0.5).to(dev)

    grids = [(scale(batch, M // 128, K // 128), SCALE_BLOCK128), (scale(batch, M), SCALE_ROW)]
    if K % 256 == 0:
        grids.append((scale(batch, M // 128, K // 256), SCALE_BLOCK_K256))
    sB2, sB3 = scale(N, K // 128), scale(batch, N, K // 128)
    for sA, modeA in grids:
        for B, sB in ((B2, sB2), (B3, sB3)):
            for combine in (COMBINE_DIV_PROD, COMBINE_MUL_PROD):
                got = {}
                try:
                    ops.GEMM_PATH = "large"
                    for persistent in (True, False):
                        ops.GEMM_PERSISTENT = persistent
                        for layout in ("rows", "columns"):
                            s = sB if layout == "rows" else sB.transpose(-1, -2).contiguous().transpose(-1, -2)
                            got[persistent, layout] = ops.gemm_i8_nt(A, B, sA, modeA, s, SCALE_ROW_K128, combine=combine)
                            want = KERNEL_PERSISTENT_CHAIN if persistent and layout == "columns" and (K // 128) % 2 == 0 else KERNEL_ONE_TILE
                            assert T.last_gemm_kernel() == want, layout
                finally:
                    ops.GEMM_PATH, ops.GEMM_PERSISTENT = "auto", True
                first = got.pop((False, "rows"))
                assert all(torch.equal(first, v) for v in got.values()), (modeA, combine)


# one wave and one workgroup per row, 8 and 16 chunks per thread; a row count that is no multiple of 4
@pytest.mark.parametrize("rows,cols", [(1, 128), (5, 4096), (130, 4224), (7, 16512), (3, 32768)])
def test_group_scales_column_by_column(T, dev, rows, cols):
    x = randn_bf16(make_gen(rows + cols), rows, cols).to(dev)
    for kw in ({}, {"clamp": False, "eps_add": True, "inv_mode": T._lib.INV_MULTIPLIER}, {"hadamard128": True}):
        q, s = T.ops.quant_row(x, group=128, **kw)
        qt, st = T.ops.quant_row(x, group=128, scale_t=True, **kw)
        assert torch.equal(q, qt) and torch.equal(s, st) and st.stride() == (1, rows)
    with pytest.raises(ValueError):
        T.ops.quant_row(x, scale_t=True)
