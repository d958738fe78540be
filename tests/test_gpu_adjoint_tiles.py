"""The warp adjoint's two tile depths (2 planes for few tiles, 4 for many) at
sizes with ragged tiles, for every interpolation and boundary: a batch of four
(4 planes) against its samples one by one (2 planes).  The flow gradient is the
same bits; a cell of the volume gradient sums some 100 rounded terms in an
order of its own, 100 x 2^-24 = 6e-6 of the largest sum."""
import pytest
import torch

from singleventriclesegmentation_amd import opticalFlow as OF
from torch_warp_ref import warp_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("boundary", [0, 1, 2])
@pytest.mark.parametrize("interpolation", [0, 1, 2])
@pytest.mark.parametrize("shape,C", [((9, 97, 103), 1), ((11, 81, 130), 3)])
def test_adjoint_tile_depths_agree(dev, shape, C, interpolation, boundary):
    g = torch.Generator(device=dev).manual_seed(3)
    nz, ny, nx = shape
    op = OF.WarpingCNN3D(OF.MeshInfo3D(nz, ny, nx, nz - 1, ny - 1, nx - 1), interpolation, boundary)
    u = torch.randn((4, C) + shape, device=dev, generator=g)
    phi = 1.5 * torch.randn((4,) + shape + (3,), device=dev, generator=g)  # some taps leave the window
    go = torch.randn((4, C) + shape, device=dev, generator=g)
    gu, gp = op.backward(u, phi, go)
    for b in range(4):
        gu1, gp1 = op.backward(u[b:b + 1].contiguous(), phi[b:b + 1].contiguous(), go[b:b + 1].contiguous())
        assert torch.equal(gp[b], gp1[0])
        assert (gu[b] - gu1[0]).abs().max().item() <= 1e-5 * gu1.abs().max().item()
    if interpolation == 2 and boundary == 1:
        # The displacement whose sum with the position is the float coordinate the op samples at.
        at = torch.stack(torch.meshgrid(*(torch.arange(n, dtype=torch.float32) for n in shape), indexing="ij")[::-1], -1)
        phi64 = ((at + phi[:1].cpu()).double() - at.double()).requires_grad_()
        u64 = u[:1].double().cpu().requires_grad_()
        r = torch.autograd.grad(warp_ref(u64, phi64), (u64, phi64), go[:1].double().cpu())
        for ours, ref in zip((gu[:1], gp[:1]), r):
            assert (ours.double().cpu() - ref).abs().max().item() <= 1e-5 * ref.abs().max().item()
