"""A decoder's first and third module are what the kernels read, whatever follows them."""
import pytest
import torch

from nglod_amd import _lib, workloads
from nglod_amd.autograd import _param_slots


@pytest.mark.parametrize("extra", [[], [torch.nn.Identity()], [torch.nn.Identity(), torch.nn.Dropout(0.0)]])
def test_decoders_with_more_modules(extra):
    net = workloads.make_model(num_lods=2, device="cpu")
    net.louts[1] = torch.nn.Sequential(*net.louts[1], *extra)
    m = net.descriptor()
    for i, l in enumerate(net.louts):
        assert (m.w0[i], m.b0[i], m.w1[i], m.b1[i]) == tuple(
            t.data_ptr() for t in (l[0].weight, l[0].bias, l[2].weight, l[2].bias))
    assert None not in [kind for kind, _ in _param_slots(net, _lib.parameter_list(net))]
