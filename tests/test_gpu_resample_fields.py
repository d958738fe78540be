"""Resampling and warping of several channels at once equals the channels one
by one, bit for bit (one channel is checked against the oracle in
test_gpu_ops.py): chunk remainders, fewer values than one chunk, chunks that
begin inside a voxel, the smallest channel count of the per-channel path."""
import pytest
import torch

from singleventriclesegmentation_amd import opticalFlow as OF

pytestmark = pytest.mark.gpu


def _mesh(shape):
    return OF.MeshInfo3D(*shape, *(float(n) for n in shape))


@pytest.mark.parametrize("boundary", [0, 1, 2])
@pytest.mark.parametrize("interpolation", [0, 1, 2])
@pytest.mark.parametrize("shape,to,C", [((4, 5, 6), (3, 7, 5), 4), ((12, 17, 9), (13, 16, 20), 5),
                                        ((9, 11, 10), (21, 4, 31), 25), ((5, 6, 7), (2, 2, 2), 3000)])
def test_prolongation_of_many_channels(dev, shape, to, C, interpolation, boundary):
    g = torch.Generator(device=dev).manual_seed(1)
    u = torch.randn(shape + (C,), device=dev, generator=g)
    op = OF.Prolongation3D(_mesh(shape), _mesh(to), interpolation, boundary)
    out = op.forwardVectorField(u)
    for c in range(0, C, max(1, C // 7)):
        assert torch.equal(out[..., c], op.forward(u[..., c].contiguous()))


@pytest.mark.parametrize("interpolation", [0, 1, 2])
def test_warp_of_a_batch_and_of_a_field(dev, interpolation):
    g = torch.Generator(device=dev).manual_seed(2)
    shape = (7, 19, 33)
    u = torch.randn((3, 2) + shape, device=dev, generator=g)
    phi = 4 * torch.randn((3,) + shape + (3,), device=dev, generator=g)
    one = OF.Warping3D(_mesh(shape), interpolation, 1)
    out = OF.WarpingCNN3D(_mesh(shape), interpolation, 1).forward(u, phi)
    field = one.forwardVectorField(u[0].permute(1, 2, 3, 0).contiguous(), phi[0])
    for b in range(3):
        for c in range(2):
            assert torch.equal(out[b, c], one.forward(u[b, c].contiguous(), phi[b]))
    for c in range(2):
        assert torch.equal(field[..., c], out[0, c])
