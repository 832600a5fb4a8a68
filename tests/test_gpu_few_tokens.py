"""dW of a step on few tokens, which rides in the launch of Y and dX on 128 x 128 tiles, against the tiled kernels: the same bits."""
import pytest
import torch

from conftest import make_gen, randn_bf16

pytestmark = pytest.mark.gpu


# one K tile and two, real tokens below and at their edges; one tile of output features beyond the few-rows kernel's 256, uneven grids
@pytest.mark.parametrize("scheme,hadamard", [("block_channel", None), ("row_block", None), ("double_channel", None), ("block_channel", 128),
                                             ("row_block", 128), ("double_channel", "full")])
@pytest.mark.parametrize("tokens,k,n", [(1, 128, 384), (16, 1024, 512), (128, 384, 1152), (129, 640, 384), (256, 128, 2048)])
def test_dw_of_few_tokens(dev, monkeypatch, tokens, k, n, scheme, hadamard):
    import triton_int8_amd as T
    if hadamard == "full":
        tokens, n = 1 << (tokens - 1).bit_length(), 512
    g = make_gen(tokens + k + n)
    X, W, dY = randn_bf16(g, tokens, k).to(dev), randn_bf16(g, n, k, std=0.02).to(dev), randn_bf16(g, tokens, n, std=1e-3).to(dev)
    x, w = X.clone().requires_grad_(True), W.clone().requires_grad_(True)
    step = T.linear_fwd_bwd(X, W, dY, scheme, hadamard)
    y = T.Int8LinearFunction.apply(x, w, None, scheme, hadamard)
    layer = (y.detach(), *torch.autograd.grad(y, (x, w), dY))
    monkeypatch.setattr(T.ops, "GEMM_PATH", "tiled")
    tiled = T.linear_fwd_bwd(X, W, dY, scheme, hadamard)
    assert torch.equal(step[2], tiled[2]) and torch.equal(layer[2], tiled[2])
    for a, b in zip(step, layer):
        assert torch.equal(a, b)
    if scheme == "double_channel":      # int32 sums: Y and dX as well
        assert torch.equal(step[0], tiled[0]) and torch.equal(step[1], tiled[1])


# workgroups of four 32 x 32 blocks: whole tiles of 64 rows and a last one of 32, a single K tile for four waves, uneven K quarters, strips
# that are and are not a multiple of 8
@pytest.mark.parametrize("m,n,k", [(64, 16384, 128), (96, 8192, 384), (160, 4224, 640), (256, 2048, 1152), (192, 5376, 256)])
@pytest.mark.parametrize("mode", ["double_channel", "block_channel", "row_block", "bias"])
def test_four_blocks_per_workgroup(dev, monkeypatch, m, n, k, mode):
    import triton_int8_amd as T
    g = make_gen(m + n + k)
    x, w = randn_bf16(g, m, k).to(dev), randn_bf16(g, n, k, std=0.02).to(dev)
    scheme = "block_channel" if mode == "bias" else mode
    layer = T.Int8Linear(k, n, bias=mode == "bias", scheme=scheme, device=dev)
    with torch.no_grad():
        layer.weight.copy_(w)
        if layer.bias is not None:
            layer.bias.copy_(randn_bf16(g, n).to(dev))
        got = layer(x)
        monkeypatch.setattr(T.ops, "GEMM_PATH", "tiled")
        want = layer(x)
    if mode == "double_channel":
        assert torch.equal(got, want)       # int32 sums
    else:
        # the same products in another order: K / 128 roundings of 2^-24 either way, then one of 2^-8 of the value to bf16 (two with a bias, of
        # values up to the product's and the bias's magnitude)
        mag = want.float().abs() + (layer.bias.detach().float().abs() if layer.bias is not None else 0.0)
        spread = (k // 128 + 4) * 2.0 ** -23 * (x.float().abs().amax(1, keepdim=True) * w.float().abs().amax() * k)
        assert bool(((got.float() - want.float()).abs() <= 2.0 ** -7 * mag + spread).all())
        assert float((got != want).float().mean()) <= 0.01


# up to 32 tokens the step's GEMMs read the weight itself: against a layer call whose weight is quantised in memory.  Fewer K tiles than waves, one
# and several batches of them per wave, uneven quarters, rows of the weight apart; the large weights of the second block of 16 tokens, as many K tiles
# per wave as Y can have (64) and about as many as dX can (57)
@pytest.mark.parametrize("scheme", ["block_channel", "double_channel"])
@pytest.mark.parametrize("tokens,k,n", [(1, 128, 384), (16, 4096, 4096), (17, 640, 1152), (31, 2176, 384), (32, 1152, 5120), (32, 14336, 4096), (20, 32768, 3328),
                                        (5, 5760, 28800)])
def test_step_from_the_weight_itself(dev, tokens, k, n, scheme):
    import triton_int8_amd as T
    from triton_int8_amd._lib import FORM_WEIGHT, last_gemm_form
    g = make_gen(tokens + k + n)
    X, dY = randn_bf16(g, tokens, k).to(dev), randn_bf16(g, tokens, n, std=1e-3).to(dev)
    W = (0.02 * torch.randn(n, k + 32, generator=torch.Generator(device=dev).manual_seed(n), device=dev)).to(torch.bfloat16)[:, 16:-16]
    W[3, 5], W[:, 7] = 1.0, 0.0
    x, w = X.clone().requires_grad_(True), W.contiguous().requires_grad_(True)
    y = T.Int8LinearFunction.apply(x, w, None, scheme, None)
    want = (y.detach(), *torch.autograd.grad(y, (x, w), dY))
    assert last_gemm_form() != FORM_WEIGHT
    step = T.linear_fwd_bwd(X, W, dY, scheme)
    assert (last_gemm_form() == FORM_WEIGHT) == (scheme == "block_channel")
    for got, a in zip(step, want):
        assert torch.equal(got, a)


def test_step_whose_outputs_are_its_inputs(dev):
    import triton_int8_amd as T
    g = make_gen(9)
    X, W, dY = randn_bf16(g, 128, 512).to(dev), randn_bf16(g, 640, 512, std=0.02).to(dev), randn_bf16(g, 128, 640, std=1e-3).to(dev)
    X[20:], dY[20:] = 0, 0
    want = T.ops.linear_step(X, W, dY, "block_channel", tokens=20)
    got = T.ops.linear_step(X, W, dY, "block_channel", tokens=20, out=(torch.empty_like(dY), X, W))
    for a, b in zip(got, want):
        assert torch.equal(a[:20] if a.shape[0] == 128 else a, b[:20] if b.shape[0] == 128 else b)


# Y and dX are computed for whole blocks of 32 rows, the last of which belong to no token: one block of 16 and two, tokens at and beside their edges; an
# infinity in X or dY reaches the padding of its 128 x 128 tiles, one in W that of its column of Y or dX, NaN none (against GEMMs on codes in memory)
@pytest.mark.parametrize("tokens", [1, 15, 16, 17, 20, 32])
@pytest.mark.parametrize("special", [None, float("inf"), float("nan")])
def test_step_rows_behind_the_tokens(dev, tokens, special):
    import triton_int8_amd as T
    from triton_int8_amd._lib import PART_BACKWARD, PART_FORWARD, PART_KEEP
    g = make_gen(tokens)
    k, n = 640, 1152
    X, W, dY = randn_bf16(g, 128, k).to(dev), randn_bf16(g, n, k, std=0.02).to(dev), randn_bf16(g, 128, n, std=1e-3).to(dev)
    if special:
        X[0, 200] = dY[0, 900] = special
        W[7, 5] = -special
        W[9] = W[:, 70] = W[40, 90] if special == float("inf") else special
    out = tuple(torch.full_like(t, 7.0) for t in (dY, X, W))
    Y, dX, dW = T.ops.linear_step(X, W, dY, "block_channel", tokens=tokens, out=out)
    wantY, _, _, saved = T.ops.linear_call(PART_FORWARD | PART_KEEP, "block_channel", None, tokens, k, n, X=X[:tokens], W=W)
    _, want_dX, want_dW, _ = T.ops.linear_call(PART_BACKWARD | PART_KEEP, "block_channel", None, tokens, k, n, X=X[:tokens], W=W, dY=dY[:tokens], saved=saved)
    for got, want in ((Y[:32], wantY[:32]), (dX[:32], want_dX[:32]), (dW, want_dW)):
        assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(nan=0.5), want.nan_to_num(nan=0.5))
    if special != float("inf"):
        assert not Y[tokens:32].any() and not dX[tokens:32].any()
    else:
        assert tokens == 32 or (Y[tokens:32].isnan().any() and dX[tokens:32].isnan().any())
