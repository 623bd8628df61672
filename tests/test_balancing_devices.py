"""The sequence-wise loss reads all layers in one launch, so layers of several
devices have to be refused before it.  Two stand-in devices on the CPU."""
import pytest
import torch

from moe_amd import balancing as Bal


def test_seq_loss_refuses_layers_of_two_devices(monkeypatch):
    monkeypatch.setattr(Bal, "_need_cuda", lambda *t: None)

    def no_launch(*args):
        raise AssertionError("launched")

    monkeypatch.setattr(Bal, "_call", no_launch)
    layers = (torch.rand(4, 8), torch.rand(4, 8, device="meta"))
    with pytest.raises(RuntimeError, match="same device"):
        Bal.seq_load_balancing_loss_func(layers, 8, 2)
