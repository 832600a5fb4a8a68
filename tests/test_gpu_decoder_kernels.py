"""RMSNorm, rotary embedding and SwiGLU kernels of the decoder layer against the expressions in float64 and the torch bf16 ones."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rel(got, want):
    got, want = got.detach().double(), want.detach().double()
    return float((got - want).norm() / want.norm())


@pytest.fixture(scope="module")
def D():
    import triton_int8_amd as T
    return T.decoder


# edges: one chunk per thread or none, the register limits (2048, 4096, 8192 elements a row), fewer rows than workgroups and more
@pytest.mark.parametrize("rows,dim", [(1, 32), (3, 2048), (7, 2080), (1023, 1024), (1025, 512), (2500, 4096), (33, 4128), (5, 8192)])
def test_rmsnorm(D, dev, rows, dim):
    gen = torch.Generator(device=dev).manual_seed(rows + dim)
    rand = lambda *s: torch.randn(*s, generator=gen, device=dev).to(torch.bfloat16)
    x, w, dy = rand(rows, dim).requires_grad_(True), (1 + 0.1 * rand(dim)).requires_grad_(True), rand(rows, dim)
    assert D._kernels_take(x, w)
    y = D._RMSNormFunction.apply(x, w, 1e-5)
    dx, dw = torch.autograd.grad(y, (x, w), dy)
    xe, we = x.detach().double().requires_grad_(True), w.detach().double().requires_grad_(True)
    ye = xe * torch.rsqrt(xe.pow(2).mean(-1, keepdim=True) + 1e-5) * we
    dxe, dwe = torch.autograd.grad(ye, (xe, we), dy.double())
    # a rounding to bf16 is off by up to 2^-9 of the value, 2^-9 / sqrt(3) in the norm; two of them in y and in dx, two in dw
    for got, want in ((y, ye), (dx, dxe), (dw, dwe)):
        assert _rel(got, want) <= 2 * 2.0 ** -9
    plain = D._rmsnorm(x, w, 1e-5)
    if dim <= 4096 and dim % 256 == 0:       # the order of the sum is that of torch's mean
        assert torch.equal(y, plain)
    for got, ours, want in zip(torch.autograd.grad(plain, (x, w), dy), (dx, dw), (dxe, dwe)):
        assert _rel(ours, want) <= 1.05 * _rel(got, want) + 1e-4          # no further from it than the torch expression
    # differentiated twice: the torch expression's graph
    g1 = torch.autograd.grad(D._RMSNormFunction.apply(x, w, 1e-5), x, dy, create_graph=True)[0]
    g0 = torch.autograd.grad(D._rmsnorm(x, w, 1e-5), x, dy, create_graph=True)[0]
    assert torch.equal(torch.autograd.grad(g1.float().sum(), w)[0], torch.autograd.grad(g0.float().sum(), w)[0])


# the smallest and largest rows and row counts that the layer hands to the kernels, steps of 256 that no power of two covers
@pytest.mark.parametrize("shape", [(8, 256), (9, 4096), (3, 5, 768), (16, 2816), (2, 1000, 1024), (1025, 3840), (4097, 512)])
def test_rmsnorm_bits(D, dev, shape):
    gen = torch.Generator(device=dev).manual_seed(sum(shape))
    rand = lambda *s: torch.randn(*s, generator=gen, device=dev).to(torch.bfloat16)
    x, dy = rand(*shape).requires_grad_(True), rand(*shape)
    norms = [D.RMSNorm(shape[-1], device=dev, fused=fused) for fused in (True, False)]
    with torch.no_grad():
        norms[0].weight.add_(0.1 * rand(shape[-1]))
        norms[1].weight.copy_(norms[0].weight)
    outs = [n(x) for n in norms]
    assert [type(y.grad_fn).__name__ == "_RMSNormFunctionBackward" for y in outs] == [True, False]
    for got, want in zip(*((y.detach(), *torch.autograd.grad(y, (x, n.weight), dy)) for y, n in zip(outs, norms))):
        assert torch.equal(got, want)


@pytest.mark.parametrize("shape", [(7, 1024), (1, 256), (64, 640), (16, 8192)])
def test_rmsnorm_sizes_left_to_the_expression(D, dev, shape):
    x = torch.randn(*shape, generator=torch.Generator(device=dev).manual_seed(1), device=dev).to(torch.bfloat16).requires_grad_(True)
    got, want = (D.RMSNorm(shape[-1], device=dev, fused=fused)(x) for fused in (True, False))
    assert torch.equal(got, want) and type(got.grad_fn) is type(want.grad_fn)


def test_rmsnorm_backward_in_a_graph(D, dev):
    gen = torch.Generator(device=dev).manual_seed(3)
    rand = lambda *s: torch.randn(*s, generator=gen, device=dev).to(torch.bfloat16)
    x, w, dy = rand(4096, 512), 1 + 0.1 * rand(512), rand(4096, 512)
    _, rstd = D.ops.rmsnorm(x, w, 1e-5)
    D.ops.rmsnorm_backward(dy, x, w, rstd)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = D.ops.rmsnorm_backward(dy, x, w, rstd)
    for _ in range(4):
        dy.copy_(rand(4096, 512))
        graph.replay()
        dx, dw = D.ops.rmsnorm_backward(dy, x, w, rstd)
        assert torch.equal(got[0], dx)
        # the same products in another order: (rows + 1) roundings of 2^-24 of their magnitudes, and one to bf16 either side
        mag = (dy.double() * x.double() * rstd.double()[:, None]).abs().sum(0)
        assert bool(((got[1].double() - dw.double()).abs() <= 2.0 ** -8 * dw.double().abs() + 4097 * 2.0 ** -23 * mag).all())
        torch.cuda.synchronize()


@pytest.mark.parametrize("batch,seq,hidden,heads,mlp", [(2, 40, 512, 8, 1024), (1, 648, 1024, 8, 2816), (2, 512, 2048, 16, 5504)])
def test_decoder_layer_bits(D, dev, monkeypatch, batch, seq, hidden, heads, mlp):
    """Output and every gradient of the layer with its kernels and with the torch expressions in their place."""
    gen = torch.Generator(device=dev).manual_seed(seq)
    layer = D.DecoderLayer(hidden, heads, mlp, device=dev)
    x = torch.randn(batch, seq, hidden, generator=gen, device=dev).to(torch.bfloat16).requires_grad_(True)
    dy = (1e-3 * torch.randn(batch, seq, hidden, generator=gen, device=dev)).to(torch.bfloat16)
    wanted = [x, *layer.parameters()]

    def outputs():
        y = layer(x)
        return [y.detach(), *torch.autograd.grad(y, wanted, dy)]
    got = outputs()
    monkeypatch.setattr(D, "_kernels_take", lambda *tensors: False)
    names = ["y", "x", *(n for n, _ in layer.named_parameters())]
    for name, a, b in zip(names, got, outputs()):
        assert torch.equal(a, b), name


# one position, the largest angles, head dims that are no power of two, an odd one, another base
@pytest.mark.parametrize("seq,dim,base", [(1, 2, 10000.0), (5, 48, 10000.0), (777, 96, 10000.0), (4097, 128, 10000.0), (70001, 64, 10000.0), (300, 33, 500000.0)])
def test_rope_tables_bits(D, dev, seq, dim, base):
    for got, want in zip(D.rope_tables(seq, dim, dev, base), D._rope_tables(seq, dim, dev, base)):
        assert got.shape == want.shape and torch.equal(got, want)


@pytest.mark.parametrize("batch,seq,heads,dim", [(1, 1, 1, 16), (2, 5, 3, 48), (3, 128, 8, 64), (1, 77, 32, 128), (2, 9, 40, 256)])
def test_rope_bits(D, dev, batch, seq, heads, dim):
    gen = torch.Generator(device=dev).manual_seed(seq)
    q, k, dq, dk = (torch.randn(batch, seq, heads, dim, generator=gen, device=dev).to(torch.bfloat16) for _ in range(4))
    q.requires_grad_(True), k.requires_grad_(True)
    cos, sin = D.rope_tables(seq, dim, dev)
    assert D._kernels_take(q, k, cos, sin)
    outs = [f(q, k, cos, sin) for f in (D._RopeFunction.apply, D._rope_pair)]
    grads = [torch.autograd.grad(o, (q, k), (dq.transpose(1, 2).contiguous().transpose(1, 2), dk)) for o in outs]
    for a, b in zip((*outs[0], *grads[0]), (*outs[1], *grads[1])):
        assert torch.equal(a, b)


@pytest.mark.parametrize("shape", [(1, 8), (3, 680), (129, 2048), (2, 17, 1024)])
def test_swiglu(D, dev, shape):
    gen = torch.Generator(device=dev).manual_seed(shape[-1])
    gate, up, d = (torch.randn(*shape, generator=gen, device=dev).mul(4).to(torch.bfloat16) for _ in range(3))
    gate.view(-1)[:4] = torch.tensor([0.0, -100.0, 100.0, -3.0e38], device=dev)
    gate.requires_grad_(True), up.requires_grad_(True)
    assert D._kernels_take(gate, up)
    out = D._SwiGLUFunction.apply(gate, up)
    got = (out, *torch.autograd.grad(out, (gate, up), d))
    plain = D._swiglu(gate, up)
    want = (plain, *torch.autograd.grad(plain, (gate, up), d))
    ge, ue = gate.detach().double().requires_grad_(True), up.detach().double().requires_grad_(True)
    exact_out = ge * torch.sigmoid(ge) * ue
    exact = (exact_out, *torch.autograd.grad(exact_out, (ge, ue), d.double()))
    for g, w, e in zip(got, want, exact):
        torch.testing.assert_close(g, w, rtol=0, atol=0, equal_nan=True)     # the bits of the torch expression
        ok = ~torch.isnan(e)
        assert _rel(g[ok], e[ok]) <= _rel(w[ok], e[ok]) + 1e-5


def test_calls_the_kernels_do_not_take(D, dev):
    x = torch.randn(4, 64, device=dev).to(torch.bfloat16)
    w = torch.nn.Parameter(torch.ones(64, device=dev, dtype=torch.bfloat16))
    assert D._kernels_take(x, w)
    assert not D._kernels_take(x.float(), w) and not D._kernels_take(x.t(), w) and not D._kernels_take(x.cpu(), w)
    assert not D._kernels_take(torch.randn(257, device=dev).to(torch.bfloat16)[1:], w)       # 2-byte aligned
    assert not D._kernels_take(x[:0], w)
    norm = D.RMSNorm(64, device=dev, fused=True)
    assert torch.equal(torch.func.vmap(norm)(x[:, None]), D.RMSNorm(64, device=dev)(x[:, None]))
    with torch.autograd.forward_ad.dual_level():
        assert not D._kernels_take(torch.autograd.forward_ad.make_dual(x, x), w)


@pytest.mark.parametrize("relayout", ["transposed", "shifted"])
def test_saved_tensors_in_another_layout(D, dev, relayout):
    """Hooks that hand a saved tensor back with other strides, or at an odd offset: the same values, so the same gradients."""
    def unpack(t):
        if relayout == "transposed":
            return t.movedim(-1, 0).contiguous().movedim(0, -1)
        return torch.cat((t.flatten()[:1], t.flatten()))[1:].view(t.shape)
    gen = torch.Generator(device=dev).manual_seed(7)
    layer = D.DecoderLayer(512, 8, 1024, device=dev)
    x = torch.randn(2, 40, 512, generator=gen, device=dev).to(torch.bfloat16).requires_grad_(True)
    wanted = [x, *layer.parameters()]
    gate, up = (torch.randn(40, 256, generator=gen, device=dev).to(torch.bfloat16).requires_grad_(True) for _ in range(2))
    q, k = (torch.randn(1, 40, 2, 64, generator=gen, device=dev).to(torch.bfloat16).requires_grad_(True) for _ in range(2))
    w = (1 + 0.1 * torch.randn(256, generator=gen, device=dev)).to(torch.bfloat16).requires_grad_(True)
    tables = D.rope_tables(40, 64, dev)
    calls = [(lambda: D._RMSNormFunction.apply(gate, w, 1e-5), (gate, w)), (lambda: D._SwiGLUFunction.apply(gate, up), (gate, up)),
             (lambda: sum(D._RopeFunction.apply(q, k, *tables)), (q, k))]
    if relayout == "shifted":        # (torch's attention wants the last dim dense)
        calls.append((lambda: layer(x), wanted))
    for call, leaves in calls:
        out = call()
        d = (1e-2 * torch.randn(*out.shape, generator=gen, device=dev)).to(torch.bfloat16)
        want = torch.autograd.grad(out, leaves, d)
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
            got = torch.autograd.grad(call(), leaves, d)
        for a, b in zip(got, want):
            assert torch.equal(a, b)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t.cpu()):
        for call, leaves in calls[:3]:
            out = call()
            with pytest.raises(RuntimeError, match="expected tensors on"):
                torch.autograd.grad(out, leaves, torch.ones_like(out))
