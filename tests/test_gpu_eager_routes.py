"""Call forms in which the direct eager route of an op must hand over to the registered custom op,
and the one-cloud FPS at its ends."""

import pytest
import torch

from torch.utils._python_dispatch import TorchDispatchMode

from gdl_amd.functional import farthest_point_sampling, segment_reduce, sort_and_build_csr
from gdl_amd.graph import SpatialGraph
from gdl_amd.se3_conv import SE3Conv

pytestmark = pytest.mark.gpu


def _graph(E=300, N=40, C=8):
    g = torch.Generator().manual_seed(0)
    col = torch.randint(0, N, (E,), generator=g)
    return torch.randn(E, C, generator=g).cuda(), sort_and_build_csr(col.cuda(), N), N


@pytest.mark.parametrize("reduce", ["sum", "mean", "max"])
def test_batched_and_recorded_gradients(reduce):
    m, csr, N = _graph()
    m.requires_grad_()
    out = segment_reduce(m, *csr, N, reduce=reduce)
    v = torch.randn(3, *out.shape, generator=torch.Generator().manual_seed(1)).cuda()
    batched, = torch.autograd.grad(out, m, v, is_grads_batched=True, retain_graph=True)
    single = [torch.autograd.grad(out, m, x, retain_graph=True)[0] for x in v]
    assert torch.equal(batched, torch.stack(single))
    # a second derivative does not exist: an error, also where another term has one
    g, = torch.autograd.grad(out.square().sum() + m.pow(3).sum(), m, create_graph=True)
    with pytest.raises(RuntimeError):
        torch.autograd.grad(g.sum(), m)


@pytest.mark.parametrize("reduce", ["sum", "mean", "max"])
def test_direct_route_equals_custom_op(reduce):
    m, csr, N = _graph()
    got = []
    for direct in (True, False):
        x = m.clone().requires_grad_()
        if direct:
            out = segment_reduce(x, *csr, N, reduce=reduce)
        else:
            with torch.device("cuda"):  # a function mode: the registered op is called
                out = segment_reduce(x, *csr, N, reduce=reduce)
        assert ("Eager" in type(out.grad_fn).__name__) is direct
        out.square().sum().backward()
        got.append((out.detach(), x.grad))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


class _Seen(TorchDispatchMode):
    """The framework's ops that pass by, as any dispatch mode sees them."""

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        if func.namespace == "geoembodied":
            self.ops.append(func._schema.name.split("::")[1])
        return func(*args, **(kwargs or {}))

    def __init__(self):
        super().__init__()
        self.ops = []


def _layer():
    g = torch.Generator().manual_seed(3)
    graph = SpatialGraph.build(torch.rand(60, 3, generator=g).cuda(), 0.4, max_num_neighbors=16)
    torch.manual_seed(4)
    layer = SE3Conv(8, 4, 8, 4).cuda()
    s = torch.randn(60, 8, generator=g).cuda().requires_grad_()
    return layer, graph, s, torch.randn(60, 4, 3, generator=g).cuda().requires_grad_()


def test_se3_conv_under_a_dispatch_mode():
    layer, graph, s, v = _layer()
    want = layer(s, v, graph)
    assert "Eager" in type(want[0].grad_fn).__name__
    wanted = [s, v, *layer.radial_basis.parameters()]
    grads = torch.autograd.grad(want[0].square().sum() + want[1].sum(), wanted)
    with _Seen() as seen:
        got = layer(s, v, graph)
        again = torch.autograd.grad(got[0].square().sum() + got[1].sum(), wanted)
    assert seen.ops == ["radial_mlp", "se3_conv_fwd", "se3_conv_bwd", "radial_mlp_bwd"]
    for a, b in zip((*got, *again), (*want, *grads)):
        assert torch.equal(a, b)


def test_se3_conv_recorded_gradients():
    layer, graph, s, v = _layer()
    out = layer(s, v, graph)[0].square().sum()
    # a second derivative does not exist: an error, also where another term has one
    g, = torch.autograd.grad(out + s.pow(3).sum(), s, create_graph=True)
    with pytest.raises(RuntimeError):
        torch.autograd.grad(g.sum(), s)


@pytest.mark.parametrize("n,k", [(0, -1), (1, 0), (1, -1), (2, 1), (500, 0), (500, 499), (500, 500)])
def test_one_cloud_fps_ends(n, k):
    pos = torch.rand(n, 3, generator=torch.Generator().manual_seed(2)).cuda()
    idx = farthest_point_sampling(pos, k)
    ref = farthest_point_sampling(pos, k, ptr=torch.tensor([0, n], device="cuda"))
    assert idx.dtype == torch.int64 and idx.numel() == max(0, min(n, k))
    assert torch.equal(idx, ref)
