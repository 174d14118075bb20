"""Farthest point sampling takes several centroids per round where the greedy order allows it: the
sequence must be the one-at-a-time one at the sizes and point sets where a round ends early."""

import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu


def _points(kind: str, n: int, seed: int) -> torch.Tensor:
    g = torch.Generator().manual_seed(seed)
    if kind == "cube":
        return torch.rand(n, 3, generator=g)
    if kind == "clumps":  # a few dense clumps far apart: the farthest points share buckets
        c = torch.randn(7, 3, generator=g) * 10
        return c[torch.randint(0, 7, (n,), generator=g)] + 0.01 * torch.randn(n, 3, generator=g)
    if kind == "lattice":  # equal distances and repeated points everywhere
        return torch.randint(0, 7, (n, 3), generator=g).float()
    if kind == "grid":  # equal distances in index order, no repeated points
        m = round(n ** (1 / 3)) + 1
        return torch.cartesian_prod(*[torch.arange(float(m))] * 3)[:n].contiguous()
    if kind == "voxel":  # a surface on a grid: ties, and more samples than distinct points
        return (torch.nn.functional.normalize(torch.randn(n, 3, generator=g), dim=1) * 16).floor()
    if kind == "line":  # boxes without volume, equal gaps
        return torch.stack([torch.randperm(n, generator=g).float(), torch.zeros(n), torch.ones(n)], 1)
    return torch.full((n, 3), 0.25)  # one point n times: every distance 0


@pytest.mark.parametrize("kind", ["cube", "clumps", "lattice", "grid", "voxel", "line", "same"])
@pytest.mark.parametrize("sizes", [[2, 63, 64, 65], [128, 129, 255, 256, 257, 383, 384, 385], [1023, 1024, 1025], [2048, 2049], [4096, 1, 130], [8192]])
def test_fps_rounds_follow_the_greedy_order(kind, sizes):
    from gdl_amd.csrc import fps_cuda
    pos = _points(kind, sum(sizes), sum(sizes))
    ptr = np.concatenate([[0], np.cumsum(sizes)])
    k = np.array([max(1, (3 * n) // 5) for n in sizes])
    got = fps_cuda(pos.cuda(), torch.from_numpy(ptr).cuda(), torch.from_numpy(k).cuda()).cpu().numpy()
    np.testing.assert_array_equal(got, oracle.fps(pos.numpy(), ptr, k))


@pytest.mark.parametrize("kind", ["cube", "clumps", "lattice", "grid", "voxel", "line", "same"])
@pytest.mark.parametrize("sizes, samples", [
    ([8193, 3], 90),            # smallest cloud of the large kernel, above the few-samples rule
    ([16384, 40], 60),          # few samples per cloud: register kernel
    ([16385, 8000, 9000], 700),  # a batch off the 64-point grid
    ([65536], 1200), ([65537], 900),      # one / two boxes per lane
    ([131073], 900), ([196608], 700),     # three, and the largest cloud
])
def test_fps_rounds_of_large_clouds(kind, sizes, samples):
    from gdl_amd.csrc import fps_cuda
    pos = _points(kind, sum(sizes), len(sizes))
    ptr = np.concatenate([[0], np.cumsum(sizes)])
    k = np.array([min(n, samples) for n in sizes])
    got = fps_cuda(pos.cuda(), torch.from_numpy(ptr).cuda(), torch.from_numpy(k).cuda()).cpu().numpy()
    np.testing.assert_array_equal(got, oracle.fps(pos.numpy(), ptr, k))


@pytest.mark.parametrize("kind", ["far groups", "all far", "inf", "nan"])
@pytest.mark.parametrize("sizes, samples", [
    ([64, 130, 700], 50), ([4096, 300], 200), ([8192], 300),
    ([9000], 60), ([9000], 300),  # register kernel, large kernel
    ([20000, 500], 300), ([70000], 200),
])
def test_distances_that_overflow_or_are_not_finite(kind, sizes, samples):
    """A bucket that no centroid can reach with a finite distance keeps all its points at +inf: the
    lowest of their indices is the next sample, wherever the bucket's order puts it."""
    from gdl_amd.csrc import fps_cuda
    n = sum(sizes)
    g = torch.Generator().manual_seed(n)
    pos = torch.rand(n, 3, generator=g)
    if kind == "far groups":  # squares overflow between the groups, not inside them
        pos = 1e18 * pos + 1e20 * torch.randint(0, 3, (n, 1), generator=g).float()
    elif kind == "all far":
        pos = 1e30 * pos
    else:
        at = torch.rand(n, generator=g) < 0.02
        pos[at, 1] = float(kind) * (torch.randint(0, 2, (int(at.sum()),), generator=g) * 2 - 1)
    ptr = np.concatenate([[0], np.cumsum(sizes)])
    k = np.array([min(m - 1, samples) for m in sizes])
    got = fps_cuda(pos.cuda(), torch.from_numpy(ptr).cuda(), torch.from_numpy(k).cuda()).cpu().numpy()
    np.testing.assert_array_equal(got, oracle.fps(pos.numpy(), ptr, k))


@pytest.mark.parametrize("n", [8193, 16384])
def test_clouds_of_the_register_kernel_need_no_workspace(n):
    from gdl_amd import _native as nat
    pos = _points("cube", n, n).cuda()
    k = 120  # above the few-samples rule
    ptr, out_ptr = torch.tensor([0, n]).cuda(), torch.tensor([0, k]).cuda()
    out = torch.empty(k, dtype=torch.int64, device="cuda")
    nat.check(nat.lib().geo_fps(nat.ptr(pos), n, nat.ptr(ptr), nat.ptr(out_ptr), 1, n, nat.ptr(out),
                                None, 0, nat.stream_of(pos.device)), "geo_fps")
    want = oracle.fps(pos.cpu().numpy(), np.array([0, n]), np.array([k]))
    np.testing.assert_array_equal(out.cpu().numpy(), want)


@pytest.mark.parametrize("counts", [[100, 3, 3, 3], [16, 200, 200, 200], [80, 80, 7, 80], [81, 0, 0, 0]])
def test_unequal_samples_of_clouds_that_the_register_kernel_holds(counts):
    """The kernel is chosen by the cloud with the most samples, which ends last."""
    from gdl_amd import _native as nat
    from gdl_amd.csrc import fps_cuda
    sizes = [8400, 300, 700, 250]
    pos = _points("cube", sum(sizes), 5)
    ptr = np.concatenate([[0], np.cumsum(sizes)])
    k = np.array(counts)
    p, kk = torch.from_numpy(ptr).cuda(), torch.from_numpy(k).cuda()
    out_ptr, info = torch.empty(5, dtype=torch.int64).cuda(), torch.empty(4, dtype=torch.int64).cuda()
    nat.check(nat.lib().geo_fps_prepare_most(nat.ptr(p), nat.ptr(kk), 4, sum(sizes), nat.ptr(out_ptr), nat.ptr(info),
                                             nat.stream_of(info.device)), "geo_fps_prepare_most")
    assert info.tolist() == [int(np.minimum(k, sizes).sum()), 8400, 0, int(np.minimum(k, sizes).max())]
    got = fps_cuda(pos.cuda(), p, kk).cpu().numpy()
    np.testing.assert_array_equal(got, oracle.fps(pos.numpy(), ptr, k))


@pytest.mark.parametrize("kind", ["cube", "lattice", "same"])
@pytest.mark.parametrize("sizes,counts", [
    ([385, 1024, 700], [1, 2, 96]), ([1025, 2048], [96, 97]), ([2049, 4096, 4095], [97, 128, 128]),
    ([4097, 8192, 8191, 500], [96, 97, 140, 3]), ([8192, 6000, 2000], [300, 2, 400]),
])
def test_few_samples(kind, sizes, counts):
    from gdl_amd.csrc import fps_cuda
    pos = _points(kind, sum(sizes), sum(counts))
    ptr = np.concatenate([[0], np.cumsum(sizes)])
    k = np.array(counts)
    got = fps_cuda(pos.cuda(), torch.from_numpy(ptr).cuda(), torch.from_numpy(k).cuda()).cpu().numpy()
    np.testing.assert_array_equal(got, oracle.fps(pos.numpy(), ptr, k))
