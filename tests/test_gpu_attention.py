"""Backward of causal attention (csrc/attention.hip) against float64 and against torch's flash kernels, whose forward it goes with."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def D():
    import triton_int8_amd as T
    return T.decoder


def _rel(got, want):
    return float((got.double() - want).norm() / want.norm())


def _exact(q, k, v, do, scale):
    q, k, v, do = (t.detach().double().contiguous() for t in (q, k, v, do))
    s = torch.matmul(q, k.transpose(2, 3).contiguous()) * scale
    p = s.masked_fill(torch.ones_like(s, dtype=torch.bool).triu(1), float("-inf")).softmax(-1)
    dp = torch.matmul(do, v.transpose(2, 3).contiguous())
    ds = p * (dp - (p * dp).sum(-1, keepdim=True)) * scale
    return torch.matmul(ds, k), torch.matmul(ds.transpose(2, 3).contiguous(), q), torch.matmul(p.transpose(2, 3).contiguous(), do)


# one row; the edges of a tile of 32 rows and of the workgroups of 128 and 256; pairs that fill the eight XCDs and that do not;
# (32, 8, 257) and (3, 100, 129) have as many workgroups of eight waves as the chip has units, the others take four
@pytest.mark.parametrize("batch,heads,seq", [(1, 1, 1), (1, 2, 31), (2, 3, 32), (1, 9, 33), (1, 8, 127), (2, 4, 129), (1, 3, 256), (1, 5, 1000),
                                             (32, 8, 257), (3, 100, 129)])
@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("layout", ["bshd", "bhsd", "sliced"])
def test_attention_backward(D, dev, batch, heads, seq, dim, layout):
    gen = torch.Generator(device=dev).manual_seed(seq + dim)

    def rand(std=1.0):
        if layout == "bhsd":
            return (std * torch.randn(batch, heads, seq, dim, generator=gen, device=dev)).to(torch.bfloat16)
        wide = 3 * dim if layout == "sliced" else dim       # a projection of q, k and v in one
        t = (std * torch.randn(batch, seq, heads, wide, generator=gen, device=dev)).to(torch.bfloat16)
        return t[..., dim:2 * dim].transpose(1, 2) if layout == "sliced" else t.transpose(1, 2)
    q, k, v = (rand().detach().requires_grad_(True) for _ in range(3))
    do, scale = rand(1e-2), 1.0 / math.sqrt(dim)
    out = D._attention(q, k, v, scale)
    assert type(out.grad_fn).__name__ == "_AttentionFunctionBackward"
    want_out = torch.nn.functional.scaled_dot_product_attention(q, k, v, is_causal=True, scale=scale)
    assert torch.equal(out, want_out)
    got, theirs = torch.autograd.grad(out, (q, k, v), do, retain_graph=True), torch.autograd.grad(want_out, (q, k, v), do)
    # the roundings of torch's kernels (two operands and the result to bf16), so no further from float64 than they are
    for name, a, b, e in zip(("dq", "dk", "dv"), got, theirs, _exact(q, k, v, do, scale)):
        if seq == 1 and name != "dv":
            assert float(a.abs().max()) <= 2.0 ** -8 * float(do.abs().max())      # the score of a single key has no gradient
            continue
        assert _rel(a, e) <= 1.01 * _rel(b, e) + 1e-4, name
    again = torch.autograd.grad(out, (q, k, v), do)
    assert all(torch.equal(a, b) for a, b in zip(got, again))


def test_attention_gradients_that_are_expanded(D, dev):
    gen = torch.Generator(device=dev).manual_seed(3)
    q, k, v = (torch.randn(2, 40, 4, 64, generator=gen, device=dev).to(torch.bfloat16).transpose(1, 2).requires_grad_(True) for _ in range(3))
    out = D._attention(q, k, v, 0.125)
    got = torch.autograd.grad(out.sum(), (q, k, v), retain_graph=True)
    for a, b in zip(got, torch.autograd.grad(out, (q, k, v), torch.ones_like(out))):
        assert torch.equal(a, b)


def test_attention_calls_left_to_torch(D, dev):
    q = torch.randn(1, 4, 64, 64, device=dev).to(torch.bfloat16).requires_grad_(True)
    wide = torch.randn(1, 4, 64, 96, device=dev).to(torch.bfloat16).requires_grad_(True)
    assert D._attention_kernels_take(q, q, q, 0.125)
    assert not D._attention_kernels_take(wide, wide, wide, 0.125) and not D._attention_kernels_take(q.float(), q.float(), q.float(), 0.125)
    assert not D._attention_kernels_take(q[..., 1:], q[..., 1:], q[..., 1:], 0.125)
    with torch.no_grad():
        assert not D._attention_kernels_take(q, q, q, 0.125)
    with torch.nn.attention.sdpa_kernel(torch.nn.attention.SDPBackend.MATH):
        assert not D._attention_kernels_take(q, q, q, 0.125)
    with torch.autocast("cuda", dtype=torch.float16):
        assert D._attention(q, q, q, 0.125).dtype == torch.float16


def test_attention_backward_in_a_graph(D, dev):
    gen = torch.Generator(device=dev).manual_seed(5)
    rand = lambda: torch.randn(2, 300, 4, 128, generator=gen, device=dev).to(torch.bfloat16).transpose(1, 2)
    q, k, v, do = (rand() for _ in range(4))
    o, lse = torch.ops.aten._scaled_dot_product_flash_attention(q, k, v, 0.0, True, False, scale=0.09)[:2]
    D.ops.attention_backward(do, q, k, v, o, lse, 0.09)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = D.ops.attention_backward(do, q, k, v, o, lse, 0.09)
    for _ in range(3):
        do.copy_(rand())
        graph.replay()
        want = D.ops.attention_backward(do, q, k, v, o, lse, 0.09)
        assert all(torch.equal(a, b) for a, b in zip(got, want))
        torch.cuda.synchronize()


# a batch, a head or a row alone, whose stride means nothing: in what comes back through autograd and in what goes in
@pytest.mark.parametrize("batch,heads,seq", [(1, 3, 40), (2, 1, 33), (2, 3, 1), (1, 1, 1)])
def test_attention_strides_of_dimensions_of_one(D, dev, batch, heads, seq):
    gen = torch.Generator(device=dev).manual_seed(11)

    def odd(t):
        return t.as_strided(t.shape, [s if n > 1 else s + 1 for n, s in zip(t.shape[:3], t.stride()[:3])] + [1], t.storage_offset())
    q, k, v, do = (torch.randn(batch, heads, seq, 64, generator=gen, device=dev).to(torch.bfloat16) for _ in range(4))
    want = torch.autograd.grad(D._attention(*(t.requires_grad_(True) for t in (q, k, v)), 0.125), (q, k, v), do)
    out = D._attention(q, k, v, 0.125)
    for a, b in zip(torch.autograd.grad(out, (q, k, v), odd(do)), want):
        assert torch.equal(a, b)
    x = [odd(t.detach()).requires_grad_(True) for t in (q, k, v)]
    out = D._attention(*x, 0.125)
    assert type(out.grad_fn).__name__ == "_AttentionFunctionBackward"
    for a, b in zip(torch.autograd.grad(out, x, do), want):
        assert torch.equal(a, b)


def test_attention_gradients_beyond_32_bit_offsets_are_torchs(D, dev):
    """The gradients' rows lie heads * head_dim apart, whatever those of q do."""
    seq = (1 << 30) // (64 * 128) - 512
    q = torch.empty((1, 64, seq + 1, 128), dtype=torch.bfloat16, device=dev).requires_grad_(True)
    assert not D._attention_kernels_take(q, q, q, 0.125)
    q = q.detach()[:, :, :seq - 1].requires_grad_(True)
    assert D._attention_kernels_take(q, q, q, 0.125)
    # more (batch, head) pairs than one call takes
    assert not D.ops.attention_backward_takes(1 << 21, 8, 16, 64) and not D.ops.attention_backward_takes(1, 8, (1 << 24) + 1, 64)
    assert D.ops.attention_backward_takes((1 << 21) - 1, 8, 16, 64)
