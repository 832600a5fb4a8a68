"""What a step leaves in its output tensors, and when."""
import ctypes

import pytest
import torch

import triton_int8_amd as T
from conftest import make_gen, randn_bf16
from triton_int8_amd import _lib, ops

pytestmark = pytest.mark.gpu


def _operands(dev, seed, m, k, n):
    g = make_gen(seed)
    return randn_bf16(g, m, k).to(dev), randn_bf16(g, n, k, std=0.02).to(dev), randn_bf16(g, m, n, std=1e-3).to(dev)


def _linear_args(X, W, dY, out, scheme, need, bias=None):
    m, k, n = X.shape[0], X.shape[1], W.shape[0]
    workspace = ops._workspace(need, X.device)
    pairs = [v for t in (X, W, dY, *out) for v in (t.data_ptr(), t.stride(0))]
    return _lib.LinearArgs(*pairs, None, None, m, k, n, ops._SCHEMES[scheme], 0, _lib.PART_FORWARD | _lib.PART_BACKWARD, 0, workspace.data_ptr(), need,
                           None, 0, None if bias is None else bias.data_ptr()), workspace


# partial maxima of one tile and of several; ragged tokens
@pytest.mark.parametrize("scheme", ["block_channel", "row_block", "double_channel"])
@pytest.mark.parametrize("tokens,k,n", [(384, 512, 640), (1001, 1152, 384), (300, 4224, 512)])
def test_quantisers_alone_leave_the_outputs(dev, scheme, tokens, k, n):
    X, W, dY = _operands(dev, tokens, tokens, k, n)
    want = T.linear_fwd_bwd(X, W, dY, scheme)
    rows = -(-tokens // 128) * 128
    before = [torch.full(s, 7.0, dtype=torch.bfloat16, device=dev) for s in ((rows, n), (rows, k), (n, k))]
    need, _ = ops._linear_sizes(tokens, k, n, scheme, None, _lib.PART_FORWARD | _lib.PART_BACKWARD, False)
    a, workspace = _linear_args(X, W, dY, before, scheme, need)
    problems, count = (_lib.GemmProblem * 3)(), ctypes.c_int(0)
    _lib.call("ti8_linear_quantise", ctypes.byref(a), problems, ctypes.byref(count), ops._stream())
    assert count.value == 3 and all(bool((t == 7.0).all()) for t in before)
    after = [torch.empty_like(t) for t in before]       # the products may go anywhere
    for p, t in zip(problems, after):
        p.C = t.data_ptr()
    _lib.call("ti8_gemm_i8_nt_multi", problems, 3, ops.GEMM_TOGETHER, ops._stream())
    for a, b in zip(after, want):
        assert torch.equal(a[:b.shape[0]], b)
    assert all(bool((t == 7.0).all()) for t in before)


# one launch for the three products and, on few tokens, another for those that the few-rows kernel takes; dX behind Y in the same memory, dW
# behind dX, and outputs beside each other in one buffer, which are none of each other's business
@pytest.mark.parametrize("scheme", ["block_channel", "double_channel"])
@pytest.mark.parametrize("m", [128, 384])
def test_outputs_that_share_memory(dev, scheme, m):
    k = n = m if m > 256 else 512
    X, W, dY = _operands(dev, m, m, k, n)
    Y, dX, dW = T.linear_fwd_bwd(X, W, dY, scheme)
    fresh = lambda: torch.full((max(m, n), k), 5.0, dtype=torch.bfloat16, device=dev)
    shared, other = fresh(), fresh()
    T.linear_fwd_bwd(X, W, dY, scheme, out=(shared[:m], shared[:m], other[:n]))
    assert torch.equal(shared[:m], dX) and torch.equal(other[:n], dW)
    shared, other = fresh(), fresh()
    T.linear_fwd_bwd(X, W, dY, scheme, out=(other[:m], shared[:m], shared[:n]))
    assert torch.equal(other[:m], Y) and torch.equal(shared[:n], dW)
    wide = torch.full((max(m, n), 3 * k), 5.0, dtype=torch.bfloat16, device=dev)
    beside = (wide[:m, :k], wide[:m, k:2 * k], wide[:n, 2 * k:])
    T.linear_fwd_bwd(X, W, dY, scheme, out=beside)
    for a, b in zip(beside, (Y, dX, dW)):
        assert torch.equal(a, b)


# the bias belongs to Y, and does not outlive it where dX or dW takes its place
@pytest.mark.parametrize("m", [128, 384])
def test_bias_of_an_output_that_is_written_over(dev, m):
    k = n = 384
    X, W, dY = _operands(dev, m, m, k, n)
    b = randn_bf16(make_gen(m), n, std=30.0).to(dev)
    Y, dX, dW = T.linear_fwd_bwd(X, W, dY, "block_channel")
    need, _ = ops._linear_sizes(m, k, n, "block_channel", None, _lib.PART_FORWARD | _lib.PART_BACKWARD, False)
    new = lambda rows: torch.empty((rows, k), dtype=torch.bfloat16, device=dev)
    shared, y, dx, dw = new(max(m, n)), new(m), new(m), new(n)
    for out, want in (((y, dx, dw), (Y + b, dX, dW)), ((shared[:m], shared[:m], dw), (dX, dX, dW)), ((shared[:m], dx, shared[:n]), (dW[:m], dX, dW))):
        a, workspace = _linear_args(X, W, dY, out, "block_channel", need, b)
        _lib.call("ti8_linear", ctypes.byref(a), ops._stream())
        for got, expected in zip(out, want):
            assert torch.equal(got[:expected.shape[0]], expected)


# rows that the product's kernel quantises itself, and nine that have a quantiser; Y over X, and Y's 32 rows over X's last one
@pytest.mark.parametrize("scheme", ["block_channel", "row_block", "double_channel"])
@pytest.mark.parametrize("tokens", [1, 3, 8, 9])
@pytest.mark.parametrize("where", ["in place", "behind"])
def test_forward_over_its_input(dev, scheme, tokens, where):
    k = n = 1024
    X, W, _ = _operands(dev, tokens, tokens, k, n)
    wq = T.linear.quantize_weight(W, scheme, None)
    want = ops.linear_call(_lib.PART_FORWARD, scheme, None, tokens, k, n, X=X, wq=wq)[0][:tokens]
    buffer = torch.zeros((256, k), dtype=torch.bfloat16, device=dev)
    x, y = buffer[:tokens], buffer[:128] if where == "in place" else buffer[tokens - 1:tokens + 127]
    x.copy_(X)
    need, _ = ops._linear_sizes(tokens, k, n, scheme, None, _lib.PART_FORWARD, True)
    workspace = ops._workspace(need, dev)
    a = _lib.LinearArgs(x.data_ptr(), k, None, 0, None, 0, y.data_ptr(), n, None, 0, None, 0, wq[0].data_ptr(), wq[1].data_ptr(), tokens, k, n,
                        ops._SCHEMES[scheme], 0, _lib.PART_FORWARD, 0, workspace.data_ptr(), need, None, 0, None)
    _lib.call("ti8_linear", ctypes.byref(a), ops._stream())
    assert torch.equal(y[:tokens], want)
