"""Modules that hold each other: each parameter once, in torch's order."""
import torch

from nglod_amd import _lib, workloads


def test_modules_that_hold_each_other():
    net = workloads.make_model(num_lods=2, device="cpu")
    holder = torch.nn.Module()
    holder.scale = torch.nn.Parameter(torch.zeros(2))
    holder.net = net
    net.holder = holder
    got = _lib.parameter_list(net)
    assert [id(p) for p in got] == [id(p) for p in net.parameters()] and len(got) == 11
