"""The autograd function on device tensors equals its host-tensor path: C_H and
gradient, for contiguous and strided densities in FP64 and FP32, and after the
context has solved another density in between."""
import numpy as np
import pytest
import torch

from fem_amd import Homogenizer
from fem_amd import workloads as W
from fem_amd.autograd import homogenize

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("strided", [False, True])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_device_path_equals_host_path(dtype, strided):
    shape = (8, 12, 10)
    rho = torch.from_numpy(W.simp_density(shape, 3, 2.0, rho_min=0.1)).to(dtype)
    if strided:
        rho = rho.permute(2, 0, 1).contiguous().permute(1, 2, 0)
    w = torch.from_numpy(np.random.default_rng(0).standard_normal((6, 6))).to(dtype)
    h = Homogenizer(shape, nu=0.3, tol=1e-11)
    got = []
    for dev in ("cpu", "cuda:0"):
        r = rho.detach().to(dev).requires_grad_(True)
        assert r.is_contiguous() != strided
        C = homogenize(r, h)
        assert C.dtype == dtype and C.device == r.device
        homogenize(torch.full(shape, 0.5, dtype=dtype, device=dev), h)  # the context moves on
        (C * w.to(dev)).sum().backward()
        assert r.grad.device == r.device
        got.append((C.detach().cpu(), r.grad.cpu()))
    h.close()
    assert torch.equal(got[0][0], got[1][0])
    assert torch.equal(got[0][1], got[1][1])


def test_wrong_size_is_refused():
    h = Homogenizer((4, 4, 4), nu=0.3)
    with pytest.raises(ValueError):
        homogenize(torch.ones((4, 4, 3), device="cuda:0"), h)
    h.close()
