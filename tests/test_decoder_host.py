"""The decoder layer's host side, as far as it needs no GPU."""
import pytest
import torch

from triton_int8_amd import Int8Linear, decoder, linear


@pytest.mark.parametrize("device", [None, "cpu", torch.device("cpu"), "meta"])
def test_rope_tables_on_every_kind_of_device(device):
    for got, want in zip(decoder.rope_tables(5, 12, device), decoder._rope_tables(5, 12, device)):
        assert got.shape == (5, 6) and got.dtype == torch.bfloat16 and got.device == want.device and (got.is_meta or torch.equal(got, want))


def test_layers_whose_call_is_more_than_the_product_stay_apart(monkeypatch):
    layers = [Int8Linear(128, n) for n in (128, 256)]
    x = torch.zeros(3, 128, dtype=torch.bfloat16, requires_grad=True)
    together = lambda: linear._one_group(x, layers)
    assert together()
    for cls, name in ((Int8Linear, "forward"), (torch.nn.Module, "__call__"), (torch.nn.Module, "_call_impl"), (Int8Linear, "__call__")):
        with monkeypatch.context() as m:
            as_written = getattr(cls, name)
            m.setattr(cls, name, lambda self, *a: as_written(self, *a))
            assert not together(), name
        assert together()
    layers[1]._call_impl = lambda y: y
    assert not together()
    del layers[1]._call_impl
    assert together()
    layers[0].compile(backend="eager")
    assert not together()
