"""The medium-size GEMM kernel (gemm_i8_mid_kernel: 128 x 128 tiles on two groups of four waves, half a K tile apart)
against the oracle: int32 path bit for bit, promotion per element within the bar of an fp32 sum in another order
(``assert_promoted_close``), over NaN-filled outputs."""
import pytest
import torch

from conftest import assert_promoted_close, bits_equal, make_gen
from oracle import double_channel_fwd32 as odf
from oracle import linear as olin

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def T():
    import triton_int8_amd
    return triton_int8_amd


@pytest.mark.parametrize("M,N,K,batch,path", [
    (128, 128, 128, 1, "tiled"),       # one K tile: the odd group has none
    (384, 256, 256, 2, "tiled"),       # two K tiles: one step, no loop; batches
    (256, 384, 384, 1, "tiled"),       # three: the last step is the odd one behind the loop, half of it empty
    (640, 896, 640, 1, "tiled"),       # five: a pair of steps and the one behind it, tile counts no multiple of 8
    (1024, 1024, 1024, 3, "tiled"),    # complete groups of tile rows, 192 tiles over three batches
    (128, 256, 32768, 1, "tiled"),     # 256 K tiles: every factor the kernel keeps
    (224, 14336, 1024, 1, "auto"),     # rows that are no multiple of 128: the last tile re-reads its last 32 rows
    (96, 14336, 14336, 1, "auto"),     # a partial tile only, which the rule sends here for its long K
    (64, 32768, 2048, 1, "auto"),      # the same for its many columns, every CU busy
    (32, 16384, 2048, 1, "few"),       # what the rule leaves to the few-rows kernel must agree with the same oracle
])
def test_medium_kernel(T, dev, monkeypatch, M, N, K, batch, path):
    from triton_int8_amd import ops
    from triton_int8_amd._lib import COMBINE_DIV_PROD, KERNEL_FEW_ROWS, KERNEL_MID, SCALE_BLOCK128, SCALE_ROW
    g = make_gen(M + 3 * N + 5 * K)
    A = torch.randint(-127, 128, (batch, M, K), generator=g, dtype=torch.int8)
    B = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8)
    pos = lambda *shape: torch.rand(*shape, generator=g) * 1e-2 + 1e-4
    nkb = K // 128
    sa_row, sb_row, sa_blk, sb_blk = pos(batch, M), pos(N), pos(batch, -(-M // 128), nkb), pos(N // 128, nkb)
    for kt in (0, 63, 64, nkb - 1):    # K tiles whose factor no other carries: a stale one shows as a large error
        if kt < nkb:
            sa_blk[:, :, kt] *= 37.0
    Ad, Bd = A.to(dev), B.to(dev)
    few = path == "few"
    monkeypatch.setattr(ops, "GEMM_PATH", "auto" if few else path)
    expected = KERNEL_FEW_ROWS if few else KERNEL_MID

    def run(*args, **kw):
        out = torch.full((batch, M, N), float("nan"), dtype=torch.bfloat16, device=dev)
        ops.gemm_i8_nt(Ad, Bd, *args, out=out, **kw)
        assert T.last_gemm_kernel() == expected
        return out

    got = run(sa_row.to(dev), SCALE_ROW, sb_row.to(dev), SCALE_ROW, acc_i32_full=True)
    acc = odf.gemm_i32(A, B)
    assert bits_equal(got, odf.dequant_epilogue(acc, sa_row, sb_row))
    got = run(sa_row.to(dev), SCALE_ROW, sb_row.to(dev), SCALE_ROW, acc_i32_full=True, post_scale=1.0 / K)
    assert bits_equal(got, (odf.dequant_epilogue(acc, sa_row, sb_row).float() * (1.0 / K)).to(torch.bfloat16))
    for sA, mA, oA, sB, mB, oB, kw in ((sa_blk, SCALE_BLOCK128, olin.BLOCK, sb_row, SCALE_ROW, olin.ROW, {}),
                                       (sa_blk, SCALE_BLOCK128, olin.BLOCK, sb_blk, SCALE_BLOCK128, olin.BLOCK, {}),
                                       (sa_row, SCALE_ROW, olin.ROW, sb_blk, SCALE_BLOCK128, olin.BLOCK, {"out_scale": 2.0 ** -7})):
        got = run(sA.to(dev), mA, sB.to(dev), mB, **kw)
        for b in (0, batch - 1):
            want, mag = olin.gemm_scaled(A[b], sA[b], oA, B, sB, oB, kw.get("out_scale"), with_magnitude=True)
            assert_promoted_close(got[b], want, mag, K, f"{M}x{N}x{K} A:{oA} B:{oB}")
    # the reference's division by the scale product: the same sums with the reciprocal scales, to the rounding of the factors
    # (one more rounding per term than the bar above allows for, so compared in the norm: K/128 + 4 roundings of 2^-24 each
    # stay below the bf16 rounding of 2^-9)
    got = run((1.0 / sa_blk).to(dev), SCALE_BLOCK128, (1.0 / sb_blk).to(dev), SCALE_BLOCK128, combine=COMBINE_DIV_PROD)
    want = run(sa_blk.to(dev), SCALE_BLOCK128, sb_blk.to(dev), SCALE_BLOCK128)
    assert float((got.double() - want.double()).norm() / want.double().norm()) <= 2.0 ** -9


def test_step_whose_gemms_take_different_kernels(T, dev):
    """1408 tokens, 2048 -> 5632: Y and dW run on 256 x 256 tiles, dX on the medium-size kernel, in one call, with the bits
    that forward and backward give when every GEMM is launched alone."""
    from conftest import randn_bf16
    g = make_gen(91)
    X, W, dY = randn_bf16(g, 1408, 2048).to(dev), randn_bf16(g, 5632, 2048, std=0.02).to(dev), randn_bf16(g, 1408, 5632, std=1e-3).to(dev)
    for scheme in ("block_channel", "double_channel"):
        Y, dX, dW = T.linear_fwd_bwd(X, W, dY, scheme)
        Y0, saved = T.linear.linear_forward(X, W, scheme)
        dX0, dW0 = T.linear.linear_backward(dY, X, W, scheme, None, saved)
        assert torch.equal(Y, Y0) and torch.equal(dX, dX0) and torch.equal(dW, dW0), scheme


# 1 to 9 K tiles (the loop takes four at a time), the longest K, batches, tile counts no multiple of 8
@pytest.mark.parametrize("M,N,K,batch", [*((256, 384, 128 * nk, 1) for nk in range(1, 10)), (128, 256, 32768, 1), (384, 1152, 1408, 3), (1024, 2048, 5632, 1)])
def test_bits_do_not_depend_on_the_kernel(T, dev, monkeypatch, M, N, K, batch):
    """Promoted sums on the medium-size kernel and on 256 x 256 tiles: the K tiles in the same order, so the same bits."""
    from triton_int8_amd import ops
    from triton_int8_amd._lib import COMBINE_DIV_PROD, KERNEL_MID, SCALE_BLOCK128, SCALE_ROW
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    A, B = (torch.randint(-127, 128, s, generator=g, dtype=torch.int8, device=dev) for s in ((batch, M, K), (N, K)))
    pos = lambda *shape: torch.rand(*shape, generator=g, device=dev) + 1e-2
    sa_row, sb_row, sa_blk, sb_blk = pos(batch, M), pos(N), pos(batch, M // 128, K // 128), pos(N // 128, K // 128)
    for sA, mA, sB, mB, kw in ((sa_blk, SCALE_BLOCK128, sb_row, SCALE_ROW, {}), (sa_blk, SCALE_BLOCK128, sb_blk, SCALE_BLOCK128, {}),
                               (sa_row, SCALE_ROW, sb_blk, SCALE_BLOCK128, {"out_scale": 2.0 ** -7}),
                               (sa_blk, SCALE_BLOCK128, sb_blk, SCALE_BLOCK128, {"combine": COMBINE_DIV_PROD})):
        outs = [torch.full((batch, M, N), float("nan"), dtype=torch.bfloat16, device=dev) for _ in range(2)]
        for path, out in zip(("tiled", "large"), outs):
            monkeypatch.setattr(ops, "GEMM_PATH", path)
            ops.gemm_i8_nt(A, B, sA, mA, sB, mB, out=out, **kw)
            assert (T.last_gemm_kernel() == KERNEL_MID) == (path == "tiled")
        assert torch.equal(*outs)
