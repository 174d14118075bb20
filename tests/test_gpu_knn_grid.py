"""Grid KNN against the exhaustive kernel, bit for bit: the grid that one workgroup builds per cloud
(clouds around its register and cell limits, empty clouds, more than 64 of them), the first step's
27 cells and the pruned shells behind it (surfaces, planes, lines, duplicates, sharply varying density,
queries far outside, non-finite coordinates)."""

import pytest
import torch

from gdl_amd.functional import knn

pytestmark = pytest.mark.gpu


def _points(kind, n, g):
    x = torch.rand(n, 3, generator=g)
    if kind == "sphere":
        x = torch.nn.functional.normalize(x - 0.5, dim=1)
    elif kind == "plane":
        x[:, 2] = 0.25
    elif kind == "line":
        x[:, 1:] = 0.5
    elif kind == "same":
        x[:] = 0.125
    elif kind == "lattice":
        x = (x * 8).floor()  # many points at the same distance
    elif kind == "density":
        x = (x - 0.5) * torch.rand(n, 1, generator=g).pow(6) * 100
    return x


def _ptr(sizes):
    return torch.tensor([0] + sizes).cumsum(0).cuda()


def _check(src, sizes, qry, qsizes, k):
    ps, pq = _ptr(sizes), _ptr(qsizes)
    idx, d = knn(qry, src, pq, ps, k)
    # empty clouds at the end leave fewer than 1024 sources per cloud: the exhaustive kernel
    more = src.shape[0] // 1024 + 1
    ref_i, ref_d = knn(qry, src, torch.cat([pq, pq[-1:].expand(more)]),
                       torch.cat([ps, ps[-1:].expand(more)]), k)
    assert torch.equal(idx, ref_i) and torch.equal(d, ref_d)


@pytest.mark.parametrize("k", [1, 2, 3, 4, 7, 8, 9, 16, 17, 32])
@pytest.mark.parametrize("kind", ["cube", "sphere", "plane", "line", "same", "lattice", "density"])
def test_kinds(kind, k):
    g = torch.Generator().manual_seed(k)
    sizes = [2048, 1, 0, 5000, 1024, 0, 1023]
    qsizes = [300, 5, 7, 201, 0, 0, 64]
    src = _points(kind, sum(sizes), g).cuda()
    qry = _points(kind, sum(qsizes), g)
    qry[::3] += torch.randn(qry[::3].shape, generator=g) * 0.1
    qry[5::50] = 40.0  # far outside
    _check(src, sizes, qry.cuda(), qsizes, k)


@pytest.mark.parametrize("sizes", [[8191], [8192], [8193], [20000, 3, 3], [81920] + [0] * 15, [81921] + [0] * 15, [1024] * 70,
                                   [16384] * 8, [16384] * 8 + [1], [70000], [16385, 16385]])
@pytest.mark.parametrize("k", [3, 16])
def test_sizes(sizes, k):
    g = torch.Generator().manual_seed(1)
    src = _points("sphere" if k == 3 else "density", sum(sizes), g).cuda()
    qsizes = [min(s, 500) for s in sizes]
    _check(src, sizes, _points("sphere", sum(qsizes), g).cuda(), qsizes, k)


@pytest.mark.parametrize("k", [3, 16])
def test_not_finite(k):
    g = torch.Generator().manual_seed(2)
    src, qry = torch.rand(6000, 3, generator=g), torch.rand(400, 3, generator=g)
    bad = torch.tensor([float("nan"), float("inf"), -float("inf"), -float("nan"), 3e38])
    for i, v in enumerate(bad):
        qry[i::40, i % 3] = v
    _check(src.cuda(), [4000, 2000], qry.cuda(), [300, 100], k)
    for i, v in enumerate(bad):
        s = src.clone()
        s[i::500, i % 3] = v
        _check(s.cuda(), [4000, 2000], qry.cuda(), [300, 100], k)
