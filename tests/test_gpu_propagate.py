"""Mask propagation in one native call equals the chains warped step by step
(Warp, whose kernel is checked against the oracle in test_gpu_ops.py), bit for
bit: one step, an odd and an even number of them, several channels, strided
flows, integer and extreme thresholds; what the native call does not take goes
step by step."""
import pytest
import torch

from singleventriclesegmentation_amd.warping import Warp, _propagate_natively, propagate

pytestmark = pytest.mark.gpu


def _by_steps(warp, a, b, fwd, bwd, threshold):
    f, r = [a], [b]
    for t in range(fwd.shape[0]):
        f.append(warp(f[-1], fwd[t:t + 1]))
        r.append(warp(r[-1], bwd[t:t + 1]))
    return tuple(torch.where(torch.cat(m) > threshold, 1.0, 0.0) for m in (f, r[::-1]))


def _inputs(dev, T, C, shape):
    g = torch.Generator(device=dev).manual_seed(T)
    masks = [(torch.rand((1, C) + shape, device=dev, generator=g) > 0.5).float() for _ in range(2)]
    return masks + [1.5 * torch.randn((T,) + shape + (3,), device=dev, generator=g) for _ in range(2)]


@pytest.mark.parametrize("T,C,shape,interpolation,threshold", [
    (1, 1, (7, 9, 33), "CUBIC_HERMITESPLINE", 0.5), (4, 1, (16, 21, 20), "CUBIC_HERMITESPLINE", 0.25),
    (5, 2, (12, 8, 30), "LINEAR", 0), (3, 3, (9, 10, 11), "NEAREST", 1), (2, 1, (5, 5, 5), "LINEAR", float("nan"))])
def test_chains_equal_steps(dev, T, C, shape, interpolation, threshold):
    warp = Warp(interpolation, "MIRROR", "numDofs", (1, 1, 1))
    args = _inputs(dev, T, C, shape)
    assert _propagate_natively(warp, *args, threshold) is not None
    for got, want in zip(propagate(warp, *args, threshold), _by_steps(warp, *args, threshold)):
        assert got.shape == (T + 1, C) + shape and torch.equal(got, want)


def test_chains_with_strided_flows_and_other_warps(dev):
    warp = Warp("CUBIC_HERMITESPLINE", "NEAREST", "numDofs", (1, 1, 1))
    a, b, fwd, bwd = _inputs(dev, 6, 1, (8, 9, 10))
    want = _by_steps(warp, a, b, fwd[::2], bwd[:1].expand(3, -1, -1, -1, -1), 0.5)
    got = propagate(warp, a, b, fwd[::2], bwd[:1].expand(3, -1, -1, -1, -1))
    assert all(torch.equal(x, y) for x, y in zip(got, want))
    swapped = fwd.permute(0, 3, 2, 1, 4).contiguous().permute(0, 3, 2, 1, 4)   # steps that are not contiguous
    assert _propagate_natively(warp, a, b, swapped, bwd, 0.5) is None
    assert _propagate_natively(lambda x, u: x, a, b, fwd, bwd, 0.5) is None
    for got, want in zip(propagate(warp, a, b, swapped, bwd), propagate(warp, a, b, fwd, bwd)):
        assert torch.equal(got, want)
    with pytest.raises(RuntimeError):
        propagate(warp, a, b.double(), fwd, bwd)
