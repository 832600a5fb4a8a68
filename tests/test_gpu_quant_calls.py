"""The quantisers of a layer call in two launches (partial maxima, conversion), against the operands quantised one by one: the same bits."""
import pytest
import torch

from conftest import make_gen, randn_bf16

pytestmark = pytest.mark.gpu


# one tile each way; parts of one tile; parts of several tiles, the last one shorter (more than 4096 rows or columns), both ways; ragged tokens;
# operands beyond the Infinity Cache, which go by the atomics form
@pytest.mark.parametrize("scheme", ["block_channel", "row_block", "double_channel"])
@pytest.mark.parametrize("tokens,k,n", [(300, 128, 384), (1001, 1152, 640), (4300, 384, 512), (290, 8320, 4224), (9000, 256, 384), (270, 13312, 13056)])
def test_step_quantised_in_two_launches(dev, monkeypatch, tokens, k, n, scheme):
    import triton_int8_amd as T
    g = torch.Generator(device=dev).manual_seed(tokens + k + n)
    rand = lambda *s: torch.randn(*s, generator=g, device=dev).to(torch.bfloat16)
    X, W, dY = rand(tokens, k), rand(n, k), rand(tokens, n)
    X[:, k // 3] *= 40.0        # maxima that sit in one column, one row, the last tile
    W[n - 1] *= 7.0
    dY[tokens - 1, n - 1] = 1e4
    X[tokens // 2, 5] = float("inf")
    got = T.linear_fwd_bwd(X, W, dY, scheme)
    x, w = X.clone().requires_grad_(True), W.clone().requires_grad_(True)
    y = T.Int8LinearFunction.apply(x, w, None, scheme, None)
    layer = (y.detach(), *torch.autograd.grad(y, (x, w), dY))
    monkeypatch.setattr(T.linear, "ONE_CALL_STEP", False)
    want = T.linear_fwd_bwd(X, W, dY, scheme)
    for name, a, b, c in zip(("Y", "dX", "dW"), got, layer, want):
        torch.testing.assert_close(a, c, rtol=0, atol=0, equal_nan=True, msg=name)
        torch.testing.assert_close(b, c, rtol=0, atol=0, equal_nan=True, msg=name)


def test_nan_is_left_out_of_partial_maxima(dev, monkeypatch):
    import triton_int8_amd as T
    g = make_gen(5)
    X, W, dY = randn_bf16(g, 400, 256).to(dev), randn_bf16(g, 384, 256).to(dev), randn_bf16(g, 400, 384).to(dev)
    X[3] = float("nan")
    W[:, 7] = float("nan")
    dY[17, 5] = float("nan")
    got = T.linear_fwd_bwd(X, W, dY, "double_channel")
    monkeypatch.setattr(T.linear, "ONE_CALL_STEP", False)
    for a, c in zip(got, T.linear_fwd_bwd(X, W, dY, "double_channel")):
        torch.testing.assert_close(a, c, rtol=0, atol=0, equal_nan=True)


@pytest.mark.parametrize("scheme", ["block_channel", "double_channel"])
@pytest.mark.parametrize("layout", ["in place", "strided"])
def test_step_into_given_outputs(dev, scheme, layout):
    """Outputs hold the partial maxima until the conversion has read them: not where they are the inputs' memory, or not dense."""
    import triton_int8_amd as T
    g = make_gen(9)
    M, K, N = 384, 640, 512
    X, W, dY = randn_bf16(g, M, K).to(dev), randn_bf16(g, N, K, std=0.02).to(dev), randn_bf16(g, M, N, std=1e-3).to(dev)
    want = T.linear_fwd_bwd(X, W, dY, scheme)
    if layout == "in place":
        out = (dY.clone(), X.clone(), W.clone())
        got = T.ops.linear_step(out[1], out[2], out[0], scheme, out=out)
    else:
        out = tuple(torch.full((r, c + 64), -3.0, dtype=torch.bfloat16, device=dev)[:, :c] for r, c in ((M, N), (M, K), (N, K)))
        got = T.ops.linear_step(X, W, dY, scheme, out=out)
        assert all(bool((torch.as_strided(o, (o.shape[0], 64), (o.stride(0), 1), o.storage_offset() + o.shape[1]) == -3.0).all()) for o in out)
    for a, b in zip(got, want):
        assert torch.equal(a, b)


# a wave per row and a workgroup per row, the longest row of either and the shortest of the next (more than 16384: a launch of its own);
# a whole step, a forward that leaves W^T behind, one that does not
@pytest.mark.parametrize("k", [4096, 4224, 16384, 16512])
@pytest.mark.parametrize("tokens", [5, 130])
def test_rows_beside_the_blocks(dev, monkeypatch, tokens, k):
    import triton_int8_amd as T
    from triton_int8_amd._lib import PART_FORWARD, PART_KEEP
    g = make_gen(tokens + k)
    n = 256
    X, W, dY = randn_bf16(g, tokens, k + 8).to(dev)[:, :k], randn_bf16(g, n, k).to(dev), randn_bf16(g, tokens, n).to(dev)
    X[tokens - 1, k - 1] = 300.0
    got = T.linear_fwd_bwd(X, W, dY, "row_block")
    forward = [T.ops.linear_call(PART_FORWARD | keep, "row_block", None, tokens, k, n, X=X, W=W)[0][:tokens] for keep in (0, PART_KEEP)]
    monkeypatch.setattr(T.linear, "ONE_CALL_STEP", False)
    for a, c in zip(got, T.linear_fwd_bwd(X, W, dY, "row_block")):
        assert torch.equal(a, c)
    assert torch.equal(forward[0], got[0]) and torch.equal(forward[1], got[0])


# a workgroup per row up to 256 rows, a wave per row beyond; the shortest and the longest row of the former and their neighbours
@pytest.mark.parametrize("rows", [1, 255, 256, 257])
@pytest.mark.parametrize("cols", [512, 640, 4096, 4224])
def test_few_rows_quantised(dev, rows, cols):
    import triton_int8_amd as T
    x = randn_bf16(make_gen(rows + cols), rows, cols + 16).to(dev)[:, :cols]
    x[rows // 2, cols - 1] = 50.0
    x[0] = 0.0
    q, s = T.ops.quant_row(x, inv_mode=T._lib.INV_AMAX_DIV_127)
    many = torch.zeros((300, cols), dtype=torch.bfloat16, device=dev)       # each row by itself: others do not change it
    many[:rows] = x
    want, scale = T.ops.quant_row(many, inv_mode=T._lib.INV_AMAX_DIV_127)
    assert torch.equal(q, want[:rows]) and torch.equal(s, scale[:rows])
    amax = x.float().abs().amax(1).clamp(min=1e-4)
    # tensors on both sides of a division: one rounding (a number over a tensor is 127 times the reciprocal to torch, two)
    scale = torch.full_like(amax, 127.0) / amax
    assert torch.equal(q.float(), torch.floor(x.float() * scale[:, None] + 0.5).clamp(-128, 127)) and torch.equal(s, amax / torch.full_like(amax, 127.0))


# rotated operands of a call in one launch: the forms of the row quantiser (up to 2048, 4096, 8192, 16384 columns, and the rows beyond that keep a launch
# of their own), tiles with missing tokens, against the separate entry points
@pytest.mark.parametrize("scheme", ["block_channel", "row_block"])
@pytest.mark.parametrize("tokens,k,n", [(1, 128, 2176), (37, 2048, 384), (130, 2176, 4096), (300, 4224, 640), (40, 512, 8320), (33, 16512, 256)])
def test_rotated_operands_in_one_launch(dev, monkeypatch, scheme, tokens, k, n):
    import triton_int8_amd as T
    g = make_gen(tokens + k + n)
    X, W, dY = randn_bf16(g, tokens, k).to(dev), randn_bf16(g, n, k, std=0.02).to(dev), randn_bf16(g, tokens, n, std=1e-3).to(dev)
    _against_entry_points(T, monkeypatch, X, W, dY, scheme, 128)


def _against_entry_points(T, monkeypatch, X, W, dY, scheme, hadamard):
    x, w = X.clone().requires_grad_(True), W.clone().requires_grad_(True)

    def results():
        y = T.Int8LinearFunction.apply(x, w, None, scheme, hadamard)
        return (*T.linear_fwd_bwd(X, W, dY, scheme, hadamard), y.detach(), *torch.autograd.grad(y, (x, w), dY))
    got = results()
    monkeypatch.setattr(T.linear, "ONE_CALL_STEP", False)
    for a, b in zip(got, results()):
        assert torch.equal(a, b)


# rotated over whole rows: lengths on either kernel, powers of two and between, one for all and all different, missing tokens, 32768 elements, and more
# than the transposed copies are made together for
@pytest.mark.parametrize("tokens,k,n", [(1, 128, 128), (200, 2944, 1152), (40, 4096, 5760), (130, 8192, 4096), (20, 32768, 128), (4100, 16384, 1024)])
def test_rotated_rows_in_one_launch(dev, monkeypatch, tokens, k, n):
    import triton_int8_amd as T
    g = make_gen(tokens + k + n)
    X, W, dY = randn_bf16(g, tokens, k).to(dev), randn_bf16(g, n, k, std=0.02).to(dev), randn_bf16(g, tokens, n, std=1e-3).to(dev)
    _against_entry_points(T, monkeypatch, X, W, dY, "double_channel", "full")
