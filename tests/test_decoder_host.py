"""The decoder layer's host side, as far as it needs no GPU."""
import pytest
import torch

from triton_int8_amd import decoder


@pytest.mark.parametrize("device", [None, "cpu", torch.device("cpu"), "meta"])
def test_rope_tables_on_every_kind_of_device(device):
    for got, want in zip(decoder.rope_tables(5, 12, device), decoder._rope_tables(5, 12, device)):
        assert got.shape == (5, 6) and got.dtype == torch.bfloat16 and got.device == want.device and (got.is_meta or torch.equal(got, want))
