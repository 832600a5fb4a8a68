"""Layers on the same input as one call: outputs and gradients against separate calls, bit for bit, and what keeps them apart."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def T():
    import triton_int8_amd
    return triton_int8_amd


def _layers(T, dev, k, features):
    layers = [T.Int8Linear(k, n, device=dev) for n in features]
    gen = torch.Generator(device=dev).manual_seed(k + sum(features))
    with torch.no_grad():
        for m in layers:
            m.weight.copy_(0.02 * torch.randn(*m.weight.shape, generator=gen, device=dev))
    return layers, gen


# one token, few rows, the last size on the few-rows kernel and the first past it, several rounds; features of one tile, as many as keep dW
# on its own launch, and different ones
@pytest.mark.parametrize("tokens,k,features", [(1, 128, (128, 128)), (37, 384, (256, 128, 640)), (256, 512, (512, 512, 512)), (257, 256, (128, 384)),
                                               (300, 1152, (384, 512, 640)), (1216, 1024, (1024, 1024, 1024)), (2048, 4096, (4096, 2816))])
def test_bits_of_separate_calls(T, dev, tokens, k, features):
    layers, gen = _layers(T, dev, k, features)
    x = torch.randn(tokens, k, generator=gen, device=dev).to(torch.bfloat16).requires_grad_(True)
    dys = [(1e-3 * torch.randn(tokens, n, generator=gen, device=dev)).to(torch.bfloat16) for n in features]
    wanted = [x, *(m.weight for m in layers)]
    ys = T.decoder._projections(x, *layers)
    assert type(ys[0].grad_fn).__name__ == "LinearGroupFunctionBackward"
    apart = [m(x) for m in layers]
    for a, b in zip((*ys, *torch.autograd.grad(ys, wanted, dys)), (*apart, *torch.autograd.grad(apart, wanted, dys))):
        assert a.shape == b.shape and torch.equal(a, b)


def test_kept_apart(T, dev):
    layers, gen = _layers(T, dev, 256, (256, 384))
    x = torch.randn(40, 256, generator=gen, device=dev).to(torch.bfloat16).requires_grad_(True)
    together = lambda x=x: type(T.decoder._projections(x, *layers)[0].grad_fn).__name__ == "LinearGroupFunctionBackward"
    assert together() and not together(x.detach()) and not together(x.t().contiguous().t())
    called = []
    hook = layers[1].register_forward_hook(lambda *a: called.append(1))
    assert not together() and called
    hook.remove()
    layers[0].weight.requires_grad_(False)
    assert not together()
    layers[0].weight.requires_grad_(True)
    layers[0].scheme = "row_block"
    assert not together()
    layers[0].scheme = "block_channel"
    assert together()
    ys = T.decoder._projections(x, *layers)
    with torch.no_grad():
        layers[0].weight.mul_(2)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(ys, x, [torch.ones_like(y) for y in ys])


# an output that nobody uses: no gradient for its weight, the others' and the input's as those of separate calls
@pytest.mark.parametrize("unused", [(0,), (2,), (0, 1)])
@pytest.mark.parametrize("tokens", [37, 300])
def test_unused_outputs(T, dev, unused, tokens):
    layers, gen = _layers(T, dev, 256, (256, 384, 640))
    x = torch.randn(tokens, 256, generator=gen, device=dev).to(torch.bfloat16).requires_grad_(True)
    dys = [(1e-3 * torch.randn(tokens, m.out_features, generator=gen, device=dev)).to(torch.bfloat16) for m in layers]
    used = [i for i in range(3) if i not in unused]
    results = []
    for ys in (T.decoder._projections(x, *layers), [m(x) for m in layers]):
        results.append(torch.autograd.grad([ys[i] for i in used], [x, *(m.weight for m in layers)], [dys[i] for i in used], allow_unused=True))
    assert [g is None for g in results[0]] == [False, *(i in unused for i in range(3))]
    for a, b in zip(*results):
        assert (a is None and b is None) or torch.equal(a, b)


@pytest.mark.parametrize("special", [float("inf"), float("nan")])
@pytest.mark.parametrize("tokens", [37, 300])
def test_non_finite_values(T, dev, special, tokens):
    layers, gen = _layers(T, dev, 384, (384, 512))
    x = torch.randn(tokens, 384, generator=gen, device=dev).to(torch.bfloat16)
    dys = [(1e-3 * torch.randn(tokens, m.out_features, generator=gen, device=dev)).to(torch.bfloat16) for m in layers]
    x[5, 130], dys[1][7, 3] = special, -special
    with torch.no_grad():
        layers[0].weight[9, 70] = special
        layers[1].weight[:, 300] = special
    x.requires_grad_(True)
    wanted = [x, *(m.weight for m in layers)]
    together, apart = T.decoder._projections(x, *layers), [m(x) for m in layers]
    assert type(together[0].grad_fn).__name__ == "LinearGroupFunctionBackward"
    for a, b in zip((*together, *torch.autograd.grad(together, wanted, dys)), (*apart, *torch.autograd.grad(apart, wanted, dys))):
        assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(nan=0.5), b.nan_to_num(nan=0.5))
