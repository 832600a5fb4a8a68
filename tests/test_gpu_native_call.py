"""The layer call made from C++ gives what the Python way gives, and leaves to it what it does not take."""
import os
import subprocess
import sys

import pytest
import torch

from conftest import ROOT

import triton_int8_amd as T
from triton_int8_amd._lib import PART_BACKWARD, PART_FORWARD, PART_KEEP

pytestmark = pytest.mark.gpu


class Named(torch.Tensor):
    pass


def _both(monkeypatch, call):
    assert T._lib.native() is not None
    made = call()
    with monkeypatch.context() as m:
        m.setattr(T._lib, "_native", False)
        plain = call()
    return made, plain


# the parts a call can have; one tile and several, whole and ragged; rows that are read in place, that begin at an odd address, that overlap
@pytest.mark.parametrize("scheme, hadamard", [("block_channel", None), ("row_block", 128), ("double_channel", None)])
@pytest.mark.parametrize("tokens", [1, 128, 300])
@pytest.mark.parametrize("rows", ["dense", "strided", "odd", "expanded"])
def test_same_results(dev, monkeypatch, scheme, hadamard, tokens, rows):
    k, n = 256, 384
    g = torch.Generator(device=dev).manual_seed(3)

    def matrix(r, c, kind="dense"):
        x = torch.randn(r, c + 8, generator=g, device=dev).to(torch.bfloat16)
        return {"dense": x[:, :c].contiguous(), "strided": x[:, :c], "odd": x[:, 1:c + 1], "expanded": x[:1, :c].expand(r, c)}[kind]

    X, W, dY, bias = matrix(tokens, k, rows), matrix(n, k), matrix(tokens, n, rows), matrix(1, n)[0]
    wq = T.linear.quantize_weight(W, scheme, hadamard)

    def call():
        Y, _, _, saved = T.ops.linear_call(PART_FORWARD | PART_KEEP, scheme, hadamard, tokens, k, n, X=X, W=W)
        keep = PART_KEEP if saved is not None else 0
        _, dX, dW, _ = T.ops.linear_call(PART_BACKWARD | keep, scheme, hadamard, tokens, k, n, X=X, W=W, dY=dY, saved=saved)
        served = T.ops.linear_call(PART_FORWARD, scheme, hadamard, tokens, k, n, X=X, wq=wq, bias=bias)[0]
        step = T.linear_fwd_bwd(X, W, dY, scheme, hadamard)
        assert Y.shape == served.shape == (-(-tokens // 128) * 128, n) and dX.shape[0] == Y.shape[0]
        return [Y[:tokens], dX[:tokens], dW, served[:tokens], *step]

    for a, b in zip(*_both(monkeypatch, call)):
        assert a.dtype == b.dtype == torch.bfloat16 and a.stride() == b.stride() and torch.equal(a, b)


@pytest.mark.parametrize("tokens", [1, 8, 9, 128, 300])
@pytest.mark.parametrize("scheme, hadamard", [("block_channel", None), ("row_block", 128)])
def test_served(dev, monkeypatch, scheme, hadamard, tokens):
    k, n = 256, 384
    X, W = torch.randn(tokens, k, device=dev).to(torch.bfloat16), torch.randn(n, k, device=dev).to(torch.bfloat16)
    wq = T.linear.quantize_weight(W, scheme, hadamard)
    want = T.ops.linear_call(PART_FORWARD, scheme, hadamard, tokens, k, n, X=X, wq=wq)[0][:tokens]
    for y in _both(monkeypatch, lambda: T.ops.linear_served(scheme, hadamard, tokens, k, n, X, wq)):
        assert y.shape == want.shape and y.stride() == want.stride() and torch.equal(y, want)
        y.resize_(tokens, n)        # the storage is what the shape needs, or more
        assert torch.equal(y, want)


@pytest.mark.filterwarnings("ignore::torch.jit.TracerWarning", "ignore:.torch.jit:DeprecationWarning")
@pytest.mark.parametrize("tokens", [3, 300])
def test_served_where_operators_are_followed(dev, tokens):
    """Y's cut to its tokens is an operator that a tracer and a dispatch mode see (the launches are not)."""
    from torch.utils._python_dispatch import TorchDispatchMode
    layer, x = T.Int8Linear(256, 384, device=dev), torch.randn(1, tokens, 256, device=dev).to(torch.bfloat16)

    class Names(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            names.append(func.overloadpacket.__name__)
            return func(*args, **(kwargs or {}))

    names = []
    with torch.no_grad():
        want = layer(x)
        assert torch.jit.trace(layer, x, check_trace=False)(x).shape == want.shape
        with Names():
            y = layer(x)
        assert torch.equal(y, want) and "slice" in names


def test_what_it_leaves_to_the_python_way(dev, monkeypatch):
    X, W = torch.randn(5, 256, device=dev).to(torch.bfloat16), torch.randn(128, 256, device=dev).to(torch.bfloat16)
    call = lambda x: T.ops.linear_call(PART_FORWARD, "block_channel", None, 5, 256, 128, X=x, W=W)[0][:5]
    want = call(X)
    assert torch.equal(call(X.as_subclass(Named)), want)
    with T._lib.timed_launches() as record:
        assert torch.equal(call(X), want)
    assert list(record) == ["ti8_linear"]
    for bad in (X.float(), X.cpu()):
        with pytest.raises(ValueError, match="X must be"):
            call(bad)
    def failing():
        with pytest.raises(T._lib.Ti8Error, match="ti8_linear failed with status .*ti8_linear") as e:
            T.ops.linear_call(PART_FORWARD, "block_channel", None, 5, 256, 128, X=X)
        return str(e.value)
    made, plain = _both(monkeypatch, failing)
    assert made == plain


def test_captured(dev):
    layer = T.Int8Linear(256, 128, device=dev)
    x = torch.randn(3, 256, device=dev).to(torch.bfloat16)
    with torch.no_grad():
        layer(x)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = layer(x)
        for seed in range(3):
            x.copy_(torch.randn(3, 256, device=dev, generator=torch.Generator(device=dev).manual_seed(seed)))
            graph.replay()
            assert torch.equal(y, layer(x))
            torch.cuda.synchronize()


ANOTHER_ALLOCATOR = """
import ctypes, os, sys
import torch
hip, made = ctypes.CDLL("libamdhip64.so"), []

@ctypes.CFUNCTYPE(ctypes.c_void_p, ctypes.c_ssize_t, ctypes.c_int, ctypes.c_void_p)
def take(size, device, stream):
    p = ctypes.c_void_p()
    assert hip.hipMalloc(ctypes.byref(p), ctypes.c_size_t(size)) == 0
    made.append(size)
    return p.value

@ctypes.CFUNCTYPE(None, ctypes.c_void_p, ctypes.c_ssize_t, ctypes.c_int, ctypes.c_void_p)
def give(p, size, device, stream):
    hip.hipFree(ctypes.c_void_p(p))

address = lambda f: ctypes.cast(f, ctypes.c_void_p).value
torch.cuda.memory.change_current_allocator(torch.cuda.memory._CUDAAllocator(torch._C._cuda_customAllocator(address(take), address(give))))
import triton_int8_amd as T
layer = T.Int8Linear(256, 128, device="cuda")
x = torch.randn(300, 256, device="cuda").bfloat16()
with torch.no_grad():
    layer(x)
    del made[:]
    layer(x)
    torch.cuda.synchronize()
    print(T._lib.native() is not None, len(made), flush=True)
os._exit(0)     # (nothing is freed behind the callbacks' end)
"""


def test_memory_comes_from_the_programs_own_allocator():
    """Y and the workspace, in a program that has put another allocator in the place of torch's before anything was allocated."""
    run = subprocess.run([sys.executable, "-c", ANOTHER_ALLOCATOR], cwd=ROOT, capture_output=True, text=True, timeout=100,
                         env={**os.environ, "PYTHONPATH": ROOT})
    assert run.returncode == 0 and run.stdout.split() == ["True", "2"], (run.returncode, run.stdout, run.stderr[-2000:])
