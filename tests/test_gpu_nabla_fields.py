"""The gradient and its adjoint of fields with any number of components equal
those of the components one by one, bit for bit (one and three components are
checked against the oracle in test_gpu_ops.py): component counts without a
kernel of their own, work-group counts that are no multiple of the 8 XCDs."""
import pytest
import torch

from singleventriclesegmentation_amd import _lib

pytestmark = pytest.mark.gpu


def _call(name, x, C, shape, out, bc):
    _lib.check(getattr(_lib.lib(), name)(_lib.ptr(x), C, *shape, 1.5, 0.75, 1.25, bc, _lib.ptr(out), _lib.stream_ptr()))
    return out


@pytest.mark.parametrize("bc", [0, 1, 2])
@pytest.mark.parametrize("shape,C", [((2, 2, 2), 2), ((5, 9, 23), 7), ((11, 17, 31), 2), ((4, 5, 6), 300)])
def test_components_one_by_one(dev, shape, C, bc):
    g = torch.Generator(device=dev).manual_seed(C)
    b = torch.randn(shape + (C,), device=dev, generator=g)
    p = torch.randn(shape + (C, 3), device=dev, generator=g)
    fwd = _call("svs_nabla3d_forward", b, C, shape, torch.empty_like(p), bc)
    bwd = _call("svs_nabla3d_backward", p, C, shape, torch.empty_like(b), bc)
    for c in range(0, C, max(1, C // 5)):
        one = b[..., c].contiguous(), p[..., c, :].contiguous()
        assert torch.equal(fwd[..., c, :], _call("svs_nabla3d_forward", one[0], 1, shape, torch.empty_like(one[1]), bc))
        assert torch.equal(bwd[..., c], _call("svs_nabla3d_backward", one[1], 1, shape, torch.empty_like(one[0]), bc))
