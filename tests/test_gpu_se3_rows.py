"""The one-node-per-row forward kernel over the channel counts it is chosen for (1, 2, 4 or 8 scalar
and 1 or 2 vector channels per lane, with and without type-2 channels) and just outside them:
bit-identical to the two-kernel path, and within float32 rounding of the float64 oracle."""

import pytest
import torch

from oracle import se3 as ose3
from test_gpu_se3 import _abi_forward, _close, _graph, _inputs

pytestmark = pytest.mark.gpu

CONFIGS = [
    # Cs, Cv, Ct, Os, Ov, Ot
    (1, 1, 1, 1, 1, 1), (15, 16, 16, 5, 3, 2), (16, 17, 0, 16, 4, 0),
    (17, 5, 2, 4, 4, 1),       # odd and above 16: not a row layer
    (18, 16, 9, 18, 5, 4), (32, 32, 0, 32, 32, 0), (30, 20, 0, 3, 17, 0),
    (36, 3, 0, 20, 3, 0), (64, 17, 5, 8, 0, 3), (60, 32, 0, 16, 16, 0),
    (68, 16, 0, 16, 16, 0), (128, 32, 0, 32, 8, 0), (100, 7, 3, 6, 0, 2), (128, 20, 16, 0, 0, 4),
    (0, 9, 4, 3, 2, 2), (8, 0, 16, 3, 0, 5),
    (7, 20, 0, 5, 4, 0), (15, 32, 3, 4, 4, 2), (32, 20, 8, 16, 16, 4), (16, 17, 0, 4, 3, 2),
    (132, 4, 0, 4, 4, 0), (16, 33, 0, 4, 4, 0), (16, 4, 17, 4, 4, 2),  # one channel too many
]


@pytest.mark.parametrize("cfg", CONFIGS, ids=[str(c) for c in CONFIGS])
@pytest.mark.parametrize("graph", ["sorted", "shuffled", "dense"])
def test_row_forward(dev, cfg, graph):
    gr = _graph(150, 1, 0.5, 100, 7, False) if graph == "dense" else \
        _graph(200, 2, 0.25, 24, sum(cfg), graph == "shuffled")
    s, v, t, W, R, bias, mask = _inputs(cfg, gr, 3, dev)
    s, v, R, mask = s.to(dev), v.to(dev), R.to(dev), mask.to(dev)
    t = t.to(dev) if t is not None else None
    bias = bias.to(dev) if bias is not None else None
    W = {k: (w.to(dev) if w is not None else None) for k, w in W.items()}
    want, Xw = _abi_forward(cfg, gr, s, v, t, W, R, bias, mask, False, True, dev)
    got, Xg = _abi_forward(cfg, gr, s, v, t, W, R, bias, mask, True, True, dev)
    for a, b in zip(list(got) + list(Xg), list(want) + list(Xw)):
        assert (a is None) == (b is None)
        assert a is None or torch.equal(a, b)
    cpu = lambda x: None if x is None else x.cpu()  # noqa: E731
    ref = ose3.se3_conv(cpu(s), cpu(v), cpu(t), cpu(gr.row), cpu(gr.col), cpu(gr.direction), cpu(gr.Y),
                        cpu(R), {k: cpu(w) for k, w in W.items()}, ose3.cg_11_2_cartesian(), cfg[3],
                        cfg[4], cfg[5], cpu(gr.avg_degree), cpu(bias), cpu(mask))
    for a, b in zip(got, ref):
        if b is not None and b.numel():
            _close(a, b, 2e-4, 2e-5)  # the bars of test_gpu_se3.py
