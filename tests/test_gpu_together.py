"""Several GEMMs of one call whose kernels are chosen for the launch as a whole, on either side of the rules, against separate calls: the
same bits, over NaN-filled outputs."""
import pytest
import torch

from conftest import make_gen

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def T():
    import triton_int8_amd
    return triton_int8_amd


def operand(g, dev, rows, k, block):
    q = torch.randint(-127, 128, (rows, k), generator=g, dtype=torch.int8).to(dev)
    s = torch.rand((rows // 128, k // 128) if block else (rows,), generator=g).add_(0.5).to(dev)
    return q, s


MID, FOUR, LARGE, CHAIN = "gemm_i8_mid_kernel", "gemm_i8_multi_kernel 128x128", "gemm_i8_multi_kernel 256x256", "gemm_i8_chain_kernel"


def check(T, dev, tokens, k, n, first, promoted, int32, i32):
    """The GEMMs of a step (first = 0) or of its backward half (1); `promoted`, `int32`: the kernel of the call's last launch."""
    from triton_int8_amd._lib import SCALE_BLOCK128, SCALE_ROW, describe_gemm_kernel
    g = make_gen(tokens + k + n)
    mode = SCALE_ROW if i32 else SCALE_BLOCK128
    problems = []
    for M, N, K in ((tokens, n, k), (tokens, k, n), (n, k, tokens))[first:]:
        (A, sA), (B, sB) = operand(g, dev, M, K, not i32), operand(g, dev, N, K, not i32)
        out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=dev)
        problems.append(dict(A=A, B=B, sA=sA, modeA=mode, sB=sB, modeB=mode, acc_i32_full=i32, out=out))
    outs = T.ops.gemm_i8_nt_multi(problems, together=True)
    kernel, _, tile = (int32 if i32 else promoted).partition(" ")
    assert describe_gemm_kernel().startswith(kernel) and tile in describe_gemm_kernel()
    for got, p in zip(outs, problems):
        assert torch.equal(got, T.ops.gemm_i8_nt(p["A"][None], p["B"], p["sA"][None], mode, p["sB"], mode, acc_i32_full=i32)[0])


# a step and its backward half: three medium-size GEMMs that stay on that kernel (19 beside 3 K tiles) or leave it, all on four waves,
# all on 256 x 256 tiles with a last round of 100 that is counted from the other end, an odd number of K tiles there (17, by lists: the whole step
# 187 us on four waves, 160 so), a long K apart
@pytest.mark.parametrize("i32", [False, True])
@pytest.mark.parametrize("tokens,k,n,first,promoted,int32", [
    (384, 1408, 2432, 0, MID, MID), (384, 1408, 2432, 1, MID, MID), (1280, 1280, 1280, 0, FOUR, FOUR), (1280, 1280, 1280, 1, MID, MID),
    (640, 2048, 5632, 0, FOUR, FOUR), (640, 2048, 5632, 1, LARGE, FOUR), (2048, 2048, 5632, 0, CHAIN, LARGE), (2048, 2048, 5632, 1, CHAIN, FOUR),
    (2176, 2048, 8192, 0, CHAIN, LARGE), (2176, 2048, 8192, 1, FOUR, FOUR), (512, 1024, 4096, 0, FOUR, FOUR), (512, 1024, 4096, 1, MID, MID)])
def test_one_kernel_for_a_step(T, dev, tokens, k, n, first, promoted, int32, i32):
    check(T, dev, tokens, k, n, first, promoted, int32, i32)


# one round of 128 x 128 tiles, 319 and 320 of them, several rounds; an odd number of K tiles in one GEMM beside the persistent kernel,
# which fills its rounds badly (10 x 32 tiles: apart) or well (16 x 16)
@pytest.mark.parametrize("i32", [False, True])
@pytest.mark.parametrize("tokens,k,n,promoted,int32", [(512, 512, 640, MID, MID), (1408, 1152, 1408, FOUR, FOUR), (2048, 1024, 1024, FOUR, FOUR),
                                                       (2048, 2048, 2048, CHAIN, LARGE), (2560, 1152, 8192, MID, FOUR), (4096, 1152, 4096, LARGE, LARGE)])
def test_a_launch_as_a_whole(T, dev, tokens, k, n, promoted, int32, i32):
    check(T, dev, tokens, k, n, 0, promoted, int32, i32)
