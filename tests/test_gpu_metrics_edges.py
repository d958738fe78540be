"""Edge lists and directed distances at sizes where their kernels can go wrong,
against SciPy's erosion and Euclidean distance transform: fewer edges than one
group of 16, more than one pass of all work-groups, squared distances beyond 31
bits, a mask of one voxel."""
import numpy as np
import pytest
import torch
from scipy import ndimage

from singleventriclesegmentation_amd import metrics

pytestmark = pytest.mark.gpu


def _sparse(shape, *points):
    m = np.zeros(shape, bool)
    for p in points:
        m[p] = True
    return m


CASES = {
    "one_voxel": ((5, 6, 7), lambda r, s: (_sparse(s, (4, 5, 6)), _sparse(s, (0, 0, 0)))),
    "fifteen_and_seventeen": ((3, 9, 40), lambda r, s: (_sparse(s, *[(1, 4, 2 * k) for k in range(15)]),
                                                        _sparse(s, *[(0, 8, 2 * k) for k in range(17)]))),
    "dense": ((64, 63, 65), lambda r, s: (r.random(s) > 0.6, r.random(s) > 0.6)),       # about 100,000 edges each
    "sparse": ((40, 50, 60), lambda r, s: (r.random(s) > 0.9999, r.random(s) > 0.999)),
    "beyond_31_bits": ((1, 2, 70000), lambda r, s: (_sparse(s, (0, 0, 0), (0, 1, 40)), _sparse(s, (0, 0, 69999)))),
}


@pytest.mark.parametrize("name", CASES)
def test_directed_distances(dev, name):
    shape, make = CASES[name]
    a, b = make(np.random.default_rng(5), shape)
    edges = [m ^ ndimage.binary_erosion(m) for m in (a, b)]
    z = [np.stack(np.nonzero(e), 1) for e in edges]

    def directed(e, f):
        if len(z[f]) < 40:  # few: exact integers
            return max(min(int(d) for d in ((z[f] - p) ** 2).sum(1)) for p in z[e].astype(np.int64))
        d = ndimage.distance_transform_edt(~edges[f])[edges[e]]
        return int(round(float((d ** 2).max())))
    t = [torch.from_numpy(m.astype(np.float32)).to(dev) for m in (a, b)]
    assert metrics.directed_hausdorff2(*t) == (directed(0, 1), directed(1, 0), len(z[0]), len(z[1]))
    assert metrics.mask_counts(*t) == (int(a.sum()), int(b.sum()), int((a & b).sum()))
    two = [torch.stack([m, m])[:, None] for m in t]
    want = (metrics.compute_dice(t[1], t[0]), metrics.compute_dice(*t), metrics.compute_hausdorff_distance(t[1], t[0]),
            metrics.compute_hausdorff_distance(*t))
    assert metrics.propagation_metrics(two[0], two[1]) == want
