"""Several GEMMs of one call whose kernels are chosen for the launch as a whole, on either side of the rules, against separate calls."""
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


# (tokens, K, N) of a step's three GEMMs: one round of 128 x 128 tiles, 319 and 320 of them, several rounds; an odd number of K tiles in
# one GEMM beside the persistent kernel, which fills its rounds badly (10 x 32 tiles) or well (16 x 16)
def check(T, dev, tokens, k, n, i32, first=0):
    from triton_int8_amd._lib import SCALE_BLOCK128, SCALE_ROW
    g = make_gen(tokens + k + n)
    mode = SCALE_ROW if i32 else SCALE_BLOCK128
    problems = []
    for M, N, K in ((tokens, n, k), (tokens, k, n), (n, k, tokens))[first:]:
        (A, sA), (B, sB) = operand(g, dev, M, K, not i32), operand(g, dev, N, K, not i32)
        problems.append(dict(A=A, B=B, sA=sA, modeA=mode, sB=sB, modeB=mode, acc_i32_full=i32))
    for got, p in zip(T.ops.gemm_i8_nt_multi(problems, together=True), problems):
        want = T.ops.gemm_i8_nt(p["A"][None], p["B"], p["sA"][None], mode, p["sB"], mode, acc_i32_full=i32)[0]
        if i32:
            assert torch.equal(got, want)
        else:
            assert float((got.double() - want.double()).norm() / want.double().norm()) < 2.0 ** -12


# a step and its backward half: three medium-size GEMMs that stay on that kernel (19 beside 3 K tiles) or leave it, all on four waves,
# all on 256 x 256 tiles with a last round of 100 that is counted from the other end, an odd number of K tiles there, a long K apart
@pytest.mark.parametrize("first", [0, 1])
@pytest.mark.parametrize("i32", [False, True])
@pytest.mark.parametrize("tokens,k,n", [(384, 1408, 2432), (1280, 1280, 1280), (640, 2048, 5632), (2048, 2048, 5632), (2176, 2048, 8192), (512, 1024, 4096)])
def test_one_kernel_for_a_step(T, dev, tokens, k, n, i32, first):
    check(T, dev, tokens, k, n, i32, first)


@pytest.mark.parametrize("i32", [False, True])
@pytest.mark.parametrize("tokens,k,n", [(512, 512, 640), (1408, 1152, 1408), (2048, 1024, 1024), (2048, 2048, 2048), (2560, 1152, 8192), (4096, 1152, 4096)])
def test_a_launch_as_a_whole(T, dev, tokens, k, n, i32):
    from triton_int8_amd._lib import SCALE_BLOCK128, SCALE_ROW
    g = make_gen(tokens + k + n)
    mode = SCALE_ROW if i32 else SCALE_BLOCK128
    problems = []
    for M, N, K in ((tokens, n, k), (tokens, k, n), (n, k, tokens)):
        (A, sA), (B, sB) = operand(g, dev, M, K, not i32), operand(g, dev, N, K, not i32)
        problems.append(dict(A=A, B=B, sA=sA, modeA=mode, sB=sB, modeB=mode, acc_i32_full=i32))
    for got, p in zip(T.ops.gemm_i8_nt_multi(problems, together=True), problems):
        want = T.ops.gemm_i8_nt(p["A"][None], p["B"], p["sA"][None], mode, p["sB"], mode, acc_i32_full=i32)[0]
        if i32:
            assert torch.equal(got, want)
        else:
            # the same products in another order: at most one bf16 rounding apart where the fp32 sums differ
            assert float((got.double() - want.double()).norm() / want.double().norm()) < 2.0 ** -12
            assert float(((got.double() - want.double()).abs() - want.double().abs() * 2.0 ** -7).max()) <= float(want.double().abs().max()) * 2.0 ** -18
