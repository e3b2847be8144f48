"""look_at on torch's default device and on every spelling of one."""
import pytest
import torch

from nglod_amd.renderer import look_at


@pytest.mark.parametrize("mode", ["persp", "ortho"])
@pytest.mark.parametrize("device", [None, "cpu", torch.device("cpu")])
def test_devices(device, mode):
    a = look_at([1.25, -0.3, 2.0], (0, 0.1, 0), 9, 5, mode=mode, fov=30.0, device=device)
    b = look_at(torch.tensor([1.25, -0.3, 2.0]), torch.tensor([0, 0.1, 0]), 9, 5, mode=mode, fov=30.0, device="cpu")
    for x, y in zip(a, b):
        assert x.shape == (45, 3) and x.device.type == "cpu" and torch.equal(x, y)
