"""The work that a user of this framework gives the GPU, as cases that can be timed and checked.

``listed()`` are the fixed cases, ``draw(rng)`` makes more of the same ranges, ``prepare`` makes what
a program holds before the call (inputs from the seed alone, the graph, CSR or layer it keeps),
``run`` is one pass through the public entry points, ``work`` the bytes and operations that pass
cannot do without, ``tolerance`` how far another correct implementation may be, and ``exact`` the
results in 64 bits from plain torch.

Kinds of case, and what each stands for:

* ``step``   a small object cloud through a whole downsampling stage: farthest point sampling, radius
             graph over the centres, CSR of its targets, sum of gathered features.  Latency counts.
* ``sample`` farthest point sampling alone: a batch of object clouds, or one lidar frame.
* ``graph``  ``SpatialGraph.build``: what every message-passing network does once per input.
* ``radius`` the radius graph of one lidar frame, most points with more neighbours than the cap.
* ``knn``    the neighbourhoods of sampled centres in their (unequal) clouds: pooling, transfer.
* ``interp`` decoder upsampling: KNN to the coarse level, inverse-distance interpolation of
             features, and its backward.
* ``reduce`` message aggregation over given edges: CSR build, segment reduction, its backward.
* ``pool``   max / mean pooling over a CSR that the program holds, forward and backward, also bf16.
* ``attend`` attention weights over the edges of a graph (softmax per target), forward and backward.
* ``conv``   one SE(3)-equivariant convolution layer on a graph that the program holds: inference,
             or forward and backward; with type-2 features or without.
"""

import math

import torch

from gdl_amd.functional import (
    farthest_point_sampling,
    knn,
    knn_interpolate,
    radius_graph,
    segment_reduce,
    segment_softmax,
    sort_and_build_csr,
)
from gdl_amd.graph import SpatialGraph
from gdl_amd.se3_conv import SE3Conv

DEV = "cuda"


def listed():
    return [
        # the smallest: one 2048-point object, sampled to 512, its graph and one feature sum
        dict(name="object_step", kind="step", n=2048, m=512, r=0.2, k=32, c=32),
        # the usual batch: 16 objects of 4096 points to 1024 centres each
        dict(name="batch_sample", kind="sample", cloud="sphere", b=16, n=4096, m=1024, ragged=False),
        # one 64-ring lidar frame to 16,384 centres: the longest serial chain
        dict(name="frame_sample", kind="sample", cloud="lidar", b=1, n=131072, m=16384, ragged=False),
        # the graph of that batch: edges, geometry, harmonics, CSR, degrees
        dict(name="batch_graph", kind="graph", b=16, n=4096, r=0.1, k=32),
        # the graph of a whole lidar frame: 5.3 M edges
        dict(name="frame_graph", kind="radius", n=131072, r=0.5, k=64),
        # 16 neighbours of a quarter of the points, clouds of unequal (odd) sizes
        dict(name="batch_knn", kind="knn", b=16, n=4096, q=1024, k=16, ragged=True),
        # decoder step of that batch: 3 nearest centres, 112 channels, with gradients
        dict(name="interp_train", kind="interp", b=16, n=4096, q=1024, k=3, c=112),
        # the largest aggregation: 4 M edges in no order, Zipf segments, half of them empty
        dict(name="reduce_large", kind="reduce", e=4194304, s=262144, c=128, op="sum", dtype="float32"),
        # pooling under mixed precision: bf16 messages, about 35 edges per target
        dict(name="pool_bf16", kind="pool", s=16384, deg=64, c=64, op="max", dtype="bfloat16"),
        # four attention heads over the batch's graph, with gradients
        dict(name="attend_train", kind="attend", b=16, n=4096, r=0.1, k=32, h=4),
        # the layer of the batch, one training pass
        dict(name="conv_train", kind="conv", b=16, n=4096, r=0.1, k=32, cs=64, cv=16, ct=0, train=True),
        # an inference pass of a layer that also carries type-2 features
        dict(name="conv_type2", kind="conv", b=16, n=2048, r=0.15, k=32, cs=32, cv=16, ct=8, train=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "sample", "sample", "graph", "radius", "knn", "interp", "reduce", "pool",
                       "attend", "conv", "conv"])
    b, n = rng.randint(1, 32), _log(rng, 300, 4096)
    r, k = round(rng.uniform(0.08, 0.25), 3), rng.choice([16, 24, 32, 48, 64])
    if kind == "step":
        n = _log(rng, 256, 8000)
        return dict(kind=kind, n=n, m=max(16, n // rng.randint(2, 8)), r=r, k=k, c=rng.choice([16, 32, 33, 64]))
    if kind == "sample":
        if rng.random() < 0.3:
            n = _log(rng, 9000, 131072)
            return dict(kind=kind, cloud="lidar", b=1, n=n, m=max(64, n // rng.randint(8, 32)), ragged=False)
        n = _log(rng, 300, 8000)
        return dict(kind=kind, cloud=rng.choice(["sphere", "cube"]), b=b, n=n,
                    m=max(16, n // rng.randint(2, 16)), ragged=rng.random() < 0.5)
    if kind == "graph":
        return dict(kind=kind, b=b, n=n, r=r, k=k)
    if kind == "radius":
        return dict(kind=kind, n=_log(rng, 4096, 131072), r=round(rng.uniform(0.3, 0.8), 3), k=k)
    if kind == "knn":
        return dict(kind=kind, b=b, n=n, q=max(8, n // rng.randint(1, 8)), k=rng.randint(2, 32),
                    ragged=rng.random() < 0.7)
    if kind == "interp":
        return dict(kind=kind, b=b, n=n, q=max(8, n // rng.randint(2, 8)), k=rng.randint(1, 8),
                    c=rng.choice([16, 33, 64, 112, 128, 160]))
    if kind in ("reduce", "pool"):
        c = rng.choice([16, 32, 33, 64, 96, 128])
        op, dt = rng.choice(["sum", "sum", "mean", "max"]), rng.choice(["float32", "float32", "bfloat16"])
        if kind == "reduce":
            e = _log(rng, 10000, 4194304)
            return dict(kind=kind, e=e, s=max(8, e // rng.randint(8, 40)), c=c, op=op, dtype=dt)
        return dict(kind=kind, s=_log(rng, 500, 40000), deg=rng.randint(8, 64), c=c, op=op, dtype=dt)
    if kind == "attend":
        return dict(kind=kind, b=b, n=n, r=r, k=k, h=rng.choice([1, 2, 4, 8]))
    cs, cv = rng.choice([(16, 8), (32, 16), (64, 16), (48, 12), (64, 32), (128, 32)])
    b = min(b, 16) if cs < 128 else min(b, 4)
    train, ct = rng.random() < 0.5, rng.choice([0, 0, 8])
    return dict(kind="conv", b=b, n=n, r=r, k=min(k, 32), cs=cs, cv=cv, ct=ct if b * n <= 32768 else 0,
                train=train)


# ── inputs ──────────────────────────────────────────────────────────


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _sizes(b, n, ragged):
    """Cloud sizes: equal, or spread over n * [0.75, 1.25] in odd steps that depend on b and n alone."""
    if not ragged:
        return [n] * b
    return [max(4, int(n * (0.75 + 0.5 * ((i * 0.618034 + 0.31) % 1.0)))) for i in range(b)]


def _ptr(sizes):
    p = [0]
    for x in sizes:
        p.append(p[-1] + x)
    return torch.tensor(p, dtype=torch.int64, device=DEV)


def _sphere(total, g):
    """Scans of object surfaces: the unit sphere with 0.01 jitter."""
    d = torch.randn(total, 3, device=DEV, generator=g)
    return d / d.norm(dim=1, keepdim=True) + 0.01 * torch.randn(total, 3, device=DEV, generator=g)


def _lidar(n, g):
    """A spinning-lidar frame in scan order: rings over -24.8 .. 2 degrees, ranges of 1 .. 80 m cut
    by the ground 1.7 m below the sensor."""
    rings = 64 if n >= 16384 else 32
    cols = -(-n // rings)
    el = torch.deg2rad(torch.linspace(-24.8, 2.0, rings, dtype=torch.float64, device=DEV))[:, None]
    az = (torch.arange(cols, dtype=torch.float64, device=DEV) * (2 * math.pi / cols))[None, :]
    rho = torch.rand(rings, cols, device=DEV, generator=g, dtype=torch.float64) * 79 + 1
    rho = rho + 0.02 * torch.randn(rings, cols, device=DEV, generator=g, dtype=torch.float64)
    hit = torch.where(el < 0, 1.7 / torch.sin(-el).clamp(min=1e-12), torch.full_like(el, math.inf))
    rho = torch.minimum(rho, hit)
    p = torch.stack([rho * torch.cos(el) * torch.cos(az), rho * torch.cos(el) * torch.sin(az),
                     rho * torch.sin(el).expand_as(rho)], dim=-1)
    return p.reshape(-1, 3)[:n].float().contiguous()


def _flip(p, g):
    """The points mirrored along a random choice of axes (no distance changes, not by a rounding)."""
    return p * (torch.randint(0, 2, (3,), device=DEV, generator=g) * 2 - 1)


def _scans(b, n, g):
    """b surface scans that depend on b and n alone, each in another order and mirrored: other inputs for
    every seed, but a graph of as many edges, so that per-edge tensors keep their shapes."""
    p = _sphere(b * n, _gen(1000003 * b + n)).reshape(b, n, 3)
    order = torch.argsort(torch.rand(b, n, device=DEV, generator=g), dim=1)
    return _flip(p.gather(1, order[..., None].expand(-1, -1, 3)).reshape(b * n, 3), g)


def _frame(n, g):
    """A lidar frame that depends on n alone, started at another azimuth and mirrored (see _scans)."""
    p, rings = _lidar(n, _gen(n)), 64 if n >= 16384 else 32
    cols = n // rings
    body = p[:rings * cols].reshape(rings, cols, 3).roll(int(torch.randint(0, cols, (1,), device=DEV, generator=g)), 1)
    return _flip(torch.cat([body.reshape(-1, 3), p[rings * cols:]]), g).contiguous()


def _cloud(case, total, g):
    if case.get("cloud") == "lidar":
        return _lidar(total, g)
    if case.get("cloud") == "cube" or case["kind"] == "step":
        return torch.rand(total, 3, device=DEV, generator=g) * 2 - 1
    return _sphere(total, g)


def _segments(case, g):
    """Targets of e edges over s segments, in no order: Zipf-like sizes capped at 64, half empty."""
    e, s = case["e"], case["s"]
    w = torch.rand(s, device=DEV, generator=g).clamp(min=1e-6).pow(-5.0).clamp(max=64.0)
    w = torch.where(torch.rand(s, device=DEV, generator=g) < 0.45, torch.zeros_like(w), w)
    edges = torch.cumsum(w.double(), 0)
    pick = torch.rand(e, device=DEV, generator=g, dtype=torch.float64) * edges[-1]
    return torch.searchsorted(edges, pick).clamp(max=s - 1)


def _dims(case):
    return case["cs"], case["cv"], case["ct"]


def _inputs(case, seed):
    """The tensors of a case, from the seed alone (also what ``exact`` starts from)."""
    g, kind = _gen(seed), case["kind"]
    if kind == "step":
        return dict(pos=_cloud(case, case["n"], g), feat=torch.randn(case["m"], case["c"], device=DEV, generator=g))
    if kind == "sample":
        sizes = _sizes(case["b"], case["n"], case["ragged"])
        return dict(pos=_cloud(case, sum(sizes), g), ptr=_ptr(sizes))
    if kind == "radius":
        return dict(pos=_frame(case["n"], g))
    if kind == "reduce":
        dt = getattr(torch, case["dtype"])
        return dict(col=_segments(case, g), msg=torch.randn(case["e"], case["c"], device=DEV, generator=g).to(dt),
                    grad=torch.randn(case["s"], case["c"], device=DEV, generator=g).to(dt))
    if kind == "pool":
        dt = getattr(torch, case["dtype"])
        deg = torch.randint(max(1, case["deg"] // 8), case["deg"] + 1, (case["s"],), device=DEV,
                            generator=torch.Generator(device=DEV).manual_seed(case["s"]))
        col = torch.repeat_interleave(torch.arange(case["s"], device=DEV), deg)
        return dict(col=col, msg=torch.randn(col.numel(), case["c"], device=DEV, generator=g).to(dt),
                    grad=torch.randn(case["s"], case["c"], device=DEV, generator=g).to(dt))
    if kind in ("knn", "interp"):
        ss = _sizes(case["b"], case["n"], case.get("ragged", False))
        qs = _sizes(case["b"], case["q"], case.get("ragged", False))
        ptr, ptr_q = _ptr(ss), _ptr(qs)
        pos = _sphere(sum(ss), g)
        # centres: a random part of each cloud
        cent = torch.cat([pos[int(o):int(o) + s][torch.randperm(s, device=DEV, generator=g)[:q]]
                          for o, s, q in zip(ptr[:-1].tolist(), ss, qs)])
        d = dict(pos=pos, ptr=ptr, cent=cent, ptr_q=ptr_q)
        if kind == "interp":
            d["feat"] = torch.randn(cent.shape[0], case["c"], device=DEV, generator=g)
            d["grad"] = torch.randn(pos.shape[0], case["c"], device=DEV, generator=g)
        return d
    b, n = case["b"], case["n"]
    d = dict(pos=_sphere(b * n, g) if kind == "conv" else _scans(b, n, g), batch=torch.arange(b, device=DEV).repeat_interleave(n), ptr=_ptr([n] * b))
    if kind == "conv":
        cs, cv, ct = _dims(case)
        d["s"] = torch.randn(b * n, cs, device=DEV, generator=g)
        d["v"] = torch.randn(b * n, cv, 3, device=DEV, generator=g)
        d["t"] = torch.randn(b * n, ct, 5, device=DEV, generator=g) if ct else None
        d["gs"] = torch.randn(b * n, cs, device=DEV, generator=g)
        d["gv"] = torch.randn(b * n, cv, 3, device=DEV, generator=g)
        d["gt"] = torch.randn(b * n, ct, 5, device=DEV, generator=g) if ct else None
    return d


def _layer(case, seed):
    """A layer with its default initialisation, drawn from the seed."""
    cs, cv, ct = _dims(case)
    with torch.random.fork_rng(devices=[]):
        torch.manual_seed(int(seed))
        conv = SE3Conv(cs, cv, cs, cv, in_type2_channels=ct, out_type2_channels=ct, radius=case["r"])
        if conv.scalar_bias is not None:
            torch.nn.init.normal_(conv.scalar_bias, std=0.1)
    return conv.to(DEV)


def _build(case, d):
    return SpatialGraph.build(d["pos"], case["r"], max_num_neighbors=case["k"], batch=d["batch"],
                              num_batch_elements=case["b"])


def prepare(case, seed):
    d, kind = _inputs(case, seed), case["kind"]
    d["case"] = case
    if kind in ("reduce", "pool", "interp"):
        name = "feat" if kind == "interp" else "msg"
        d[name].requires_grad_(True)
    if kind == "pool":
        d["csr"] = sort_and_build_csr(d["col"], case["s"])
    if kind == "attend":
        d["graph"] = _build(case, d)
        g = _gen(seed + 1)
        d["scores"] = torch.randn(d["graph"].E, case["h"], device=DEV, generator=g).requires_grad_(True)
        d["grad"] = torch.randn(d["graph"].E, case["h"], device=DEV, generator=g)
    if kind == "conv":
        d["graph"] = _build(case, d)
        d["conv"] = _layer(case, seed)
        if case["train"]:
            for x in ("s", "v", "t"):
                if d[x] is not None:
                    d[x].requires_grad_(True)
    return d


# ── one pass ────────────────────────────────────────────────────────


def run(state):
    case = state["case"]
    return _RUN[case["kind"]](state, case)


def _run_step(st, case):
    idx = farthest_point_sampling(st["pos"], case["m"])
    cent = st["pos"][idx]
    row, col = radius_graph(cent, case["r"], max_num_neighbors=case["k"])
    csr = sort_and_build_csr(col, case["m"])
    return idx, segment_reduce(st["feat"][row], *csr, case["m"])


def _run_sample(st, case):
    if case["b"] == 1:
        return farthest_point_sampling(st["pos"], case["m"])
    return farthest_point_sampling(st["pos"], case["m"], ptr=st["ptr"])


def _run_graph(st, case):
    g = _build(case, st)
    return dict(row=g.row, col=g.col, direction=g.direction, dist=g.dist, col_sorted=g.col_sorted,
                perm=g.perm, node_start=g.node_start, node_end=g.node_end, Y=g.Y, avg_degree=g.avg_degree)


def _run_radius(st, case):
    return radius_graph(st["pos"], case["r"], max_num_neighbors=case["k"])


def _run_knn(st, case):
    return knn(st["cent"], st["pos"], st["ptr_q"], st["ptr"], case["k"])


def _run_interp(st, case):
    st["feat"].grad = None
    idx, dist = knn(st["pos"], st["cent"], st["ptr"], st["ptr_q"], case["k"])
    out = knn_interpolate(st["feat"], idx, dist)
    out.backward(st["grad"])
    return out.detach(), st["feat"].grad


def _run_reduce(st, case):
    st["msg"].grad = None
    csr = sort_and_build_csr(st["col"], case["s"])
    out = segment_reduce(st["msg"], *csr, case["s"], reduce=case["op"])
    out.backward(st["grad"])
    return out.detach(), st["msg"].grad


def _run_pool(st, case):
    st["msg"].grad = None
    out = segment_reduce(st["msg"], *st["csr"], case["s"], reduce=case["op"])
    out.backward(st["grad"])
    return out.detach(), st["msg"].grad


def _run_attend(st, case):
    st["scores"].grad = None
    g = st["graph"]
    w = segment_softmax(st["scores"], g.perm, g.node_start, g.node_end, g.N, contiguous_csr=True)
    w.backward(st["grad"])
    return w.detach(), st["scores"].grad


def _run_conv(st, case):
    conv, graph = st["conv"], st["graph"]
    if not case["train"]:
        with torch.no_grad():
            return tuple(conv(st["s"], st["v"], graph, type2=st["t"]))
    conv.zero_grad(set_to_none=True)
    feats = [st[x] for x in ("s", "v", "t") if st[x] is not None]
    for x in feats:
        x.grad = None
    outs = conv(st["s"], st["v"], graph, type2=st["t"])
    torch.autograd.backward(outs, [st[x] for x in ("gs", "gv", "gt") if st[x] is not None])
    return dict(out=[x.detach() for x in outs], feat=[x.grad for x in feats],
                weight=[p.grad for p in conv.parameters()])


_RUN = dict(step=_run_step, sample=_run_sample, graph=_run_graph, radius=_run_radius, knn=_run_knn,
            interp=_run_interp, reduce=_run_reduce, pool=_run_pool, attend=_run_attend, conv=_run_conv)


# ── what a pass cannot do without ───────────────────────────────────


def _edges(case):
    """Expected edges of a graph on sphere clouds: a cap of radius r holds n r^2 / 4 points."""
    return case["b"] * case["n"] * min(case["k"], case["n"] * case["r"] ** 2 / 4)


def work(case):
    kind = case["kind"]
    if kind == "step":
        e = case["m"] * min(case["k"], case["m"] * (4.19 / 8) * case["r"] ** 3)
        return {"bytes": case["n"] * 12 + case["m"] * (8 + 8 * case["c"]) + e * 16,
                "flops": 8 * case["n"] + e * (8 + case["c"])}
    if kind == "sample":
        n, m = sum(_sizes(case["b"], case["n"], case["ragged"])), case["b"] * case["m"]
        return {"bytes": n * 12 + m * 8, "flops": 8 * n}
    if kind == "graph":
        e, n = _edges(case), case["b"] * case["n"]
        return {"bytes": n * (12 + 8 + 12) + e * (16 + 8 + 13 * 4), "flops": e * 50}
    if kind == "radius":
        e = case["n"] * case["k"] * 0.6
        return {"bytes": case["n"] * 12 + e * 16, "flops": e * 8}
    if kind in ("knn", "interp"):
        n = sum(_sizes(case["b"], case["n"], case.get("ragged", False)))
        q = sum(_sizes(case["b"], case["q"], case.get("ragged", False)))
        if kind == "knn":
            return {"bytes": (n + q) * 12 + q * case["k"] * 12, "flops": q * case["k"] * 8}
        c, k = case["c"], case["k"]
        return {"bytes": (n + q) * 12 + (q + n) * c * 4 + n * c * 4 + q * c * 4, "flops": n * k * (8 + 4 * c)}
    if kind in ("reduce", "pool"):
        b = 2 if case["dtype"] == "bfloat16" else 4
        e = case["e"] if kind == "reduce" else int(case["s"] * case["deg"] * 0.5625)
        s, c = case["s"], case["c"]
        moved = 2 * (e + s) * c * b + (4 * s * c if case["op"] == "max" else 0)
        return {"bytes": moved + (e * 8 + s * 8 if kind == "reduce" else s * 8), "flops": e * c}
    e, n = _edges(case), case["b"] * case["n"]
    if kind == "attend":
        return {"bytes": e * case["h"] * 4 * 4 + n * 8, "flops": e * case["h"] * 8}
    cs, cv, ct = _dims(case)
    w, paths = cs + 3 * cv + 5 * ct, 9 if ct else 5
    agg = (cs + cv + ct) * cs + 3 * (cs + 2 * cv) * cv + 5 * (cs + cv + ct) * ct
    x = (cs + cv + ct) + 3 * (cs + 2 * cv) + 5 * (cs + cv + ct if ct else 0)
    radial = 2 * (16 * 64 + 64 * paths)
    fwd_b = n * 2 * w * 4 + e * (8 + 4 + 12 + (36 if ct else 4)) + n * 12
    fwd_f = n * 2 * agg + e * (2 * x + radial)
    if not case["train"]:
        return {"bytes": fwd_b, "flops": fwd_f}
    return {"bytes": 2 * fwd_b + n * 2 * w * 4, "flops": 3 * fwd_f}


# What another correct implementation may differ by: float32 sums in another order, about four times the
# distance from 64-bit results that was seen over these ranges (bfloat16: its roundings of the results).
def tolerance(case):
    kind = case["kind"]
    if kind in ("sample", "radius", "knn"):
        return "exact"
    if kind in ("step", "graph"):
        return {"rel": 4e-7, "max": 4e-6}
    if kind in ("reduce", "pool"):
        if case["dtype"] == "bfloat16":
            return {"rel": 7e-3, "max": 1.6e-2}
        return {"rel": 6e-7, "max": 1e-5}
    if kind in ("interp", "attend"):
        return {"rel": 4e-7, "max": 1e-5}
    return {"rel": 6e-6, "max": 4e-5}


# ── the results in 64 bits ──────────────────────────────────────────


def _d32(a, b):
    """Squared distances as the framework defines them: every operation rounded to float32."""
    d = [a[:, None, i] - b[None, :, i] for i in range(3)]
    return (d[0] * d[0] + d[1] * d[1]) + d[2] * d[2]


def _nearest(q, s, k):
    """The k nearest of s to each of q by (distance, index): indices and float32 distances."""
    idx, dist = [], []
    for at in range(0, q.shape[0], 1024):
        d, i = torch.sort(_d32(q[at:at + 1024], s), dim=1, stable=True)
        idx.append(i[:, :k])
        dist.append(d[:, :k])
    return torch.cat(idx), torch.cat(dist)


def _plain_graph(pos, ptr, r, k):
    """Radius graph by brute force: (row, col), targets ascending, sources ascending."""
    r2 = torch.tensor(float(r) * float(r), dtype=torch.float32, device=DEV)
    rows, cols = [], []
    p = ptr.tolist()
    for lo, hi in zip(p[:-1], p[1:]):
        x = pos[lo:hi]
        i, d = _nearest(x, x, min(k + 1, hi - lo))
        me = torch.arange(hi - lo, device=DEV)[:, None]
        ok = (d < r2) & (i != me)
        ok &= torch.cumsum(ok, 1) <= k
        src = torch.sort(torch.where(ok, i, hi - lo), dim=1).values
        keep = src < hi - lo
        rows.append(src[keep] + lo)
        cols.append(me.expand_as(src)[keep] + lo)
    return torch.cat(rows), torch.cat(cols)


def _geometry(pos, row, col):
    x = pos.double()
    diff = x[col] - x[row]
    dist = diff.norm(dim=1).clamp(min=1e-8)
    u = diff / dist[:, None]
    return u, dist, _harmonics(u)


def _harmonics(u):
    x, y, z = u[:, 0], u[:, 1], u[:, 2]
    c1, c2 = math.sqrt(3 / (4 * math.pi)), math.sqrt(15 / (4 * math.pi))
    return torch.stack([torch.full_like(x, math.sqrt(1 / (4 * math.pi))), c1 * y, c1 * z, c1 * x, c2 * x * y,
                        c2 * y * z, math.sqrt(5 / (16 * math.pi)) * (3 * z * z - 1), c2 * x * z,
                        0.5 * c2 * (x * x - y * y)], dim=1)


def _average_degree(row, col, n, b):
    per = torch.bincount(col, minlength=n).reshape(b, -1).double().mean(dim=1)
    return per.clamp(min=1.0).repeat_interleave(n // b)


def _reduce64(msg, col, s, op):
    c = msg.shape[1]
    if op == "max":
        out = torch.zeros(s, c, dtype=torch.float64, device=DEV)
        return out.scatter_reduce(0, col[:, None].expand(-1, c), msg, "amax", include_self=False)
    out = torch.zeros(s, c, dtype=torch.float64, device=DEV).index_add(0, col, msg)
    if op == "mean":
        out = out / torch.bincount(col, minlength=s).clamp(min=1)[:, None].double()
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind in ("sample", "radius"):
        return None  # indices only
    d = _inputs(case, seed)
    if kind == "step":
        pos = d["pos"]  # the greedy selection in plain torch, then its graph
        near, idx = _d32(pos, pos[:1])[:, 0], [torch.zeros((), dtype=torch.int64, device=DEV)]
        for _ in range(case["m"] - 1):
            i = (near == near.max()).to(torch.uint8).argmax()
            idx.append(i)
            near = torch.minimum(near, _d32(pos, pos[i][None])[:, 0])
        cent = pos[torch.stack(idx)]
        row, col = _plain_graph(cent, _ptr([case["m"]]), case["r"], case["k"])
        return None, _reduce64(d["feat"].double()[row], col, case["m"], "sum")
    if kind == "graph":
        row, col = _plain_graph(d["pos"], d["ptr"], case["r"], case["k"])
        u, dist, y = _geometry(d["pos"], row, col)
        return dict(row=None, col=None, direction=u, dist=dist, col_sorted=None, perm=None, node_start=None,
                    node_end=None, Y=y, avg_degree=_average_degree(row, col, d["pos"].shape[0], case["b"]))
    if kind in ("knn", "interp"):
        swap = kind == "interp"
        q, s, pq, ps = (d["pos"], d["cent"], d["ptr"], d["ptr_q"]) if swap else (d["cent"], d["pos"], d["ptr_q"], d["ptr"])
        k, idx, dist = case["k"], [], []
        for a, b, lo, hi in zip(pq[:-1].tolist(), pq[1:].tolist(), ps[:-1].tolist(), ps[1:].tolist()):
            i, _ = _nearest(q[a:b], s[lo:hi], k)
            w = (q[a:b, None].double() - s[lo:hi][i].double()).pow(2).sum(-1)
            short = k - i.shape[1]
            idx.append(torch.nn.functional.pad(i + lo, (0, short), value=-1))
            dist.append(torch.nn.functional.pad(w, (0, short), value=1e30))
        idx, dist = torch.cat(idx), torch.cat(dist)
        if kind == "knn":
            return None, dist
        feat = d["feat"].double().requires_grad_(True)
        w = torch.where(idx >= 0, dist.clamp(min=1e-4).rsqrt(), torch.zeros_like(dist))
        w = w / w.sum(dim=1, keepdim=True).clamp(min=1e-8)
        out = sum(w[:, j, None] * feat[idx[:, j].clamp(min=0)] for j in range(k))
        out.backward(d["grad"].double())
        return out.detach(), feat.grad
    if kind in ("reduce", "pool"):
        if d["msg"].numel() > 1 << 30:
            return None
        msg = d["msg"].double().requires_grad_(True)
        out = _reduce64(msg, d["col"], case["s"], case["op"])
        if case["op"] != "max":
            out.backward(d["grad"].double())
            return out.detach(), msg.grad
        with torch.no_grad():  # the gradient shared evenly by tied maxima
            hit = (msg == out[d["col"]]).double()
            ties = torch.zeros_like(out).index_add(0, d["col"], hit)
            return out.detach(), hit * (d["grad"].double() / ties.clamp(min=1))[d["col"]]
    row, col = _plain_graph(d["pos"], d["ptr"], case["r"], case["k"])
    n = d["pos"].shape[0]
    if kind == "attend":
        g = _gen(seed + 1)
        x = torch.randn(col.numel(), case["h"], device=DEV, generator=g).double().requires_grad_(True)
        gw = torch.randn(col.numel(), case["h"], device=DEV, generator=g).double()
        at = col[:, None].expand(-1, case["h"])
        top = torch.full((n, case["h"]), -math.inf, dtype=torch.float64, device=DEV).scatter_reduce(
            0, at, x.detach(), "amax")
        ex = (x - top[col]).exp()
        w = ex / torch.zeros_like(top).index_add(0, col, ex).clamp(min=1e-8)[col]
        w.backward(gw)
        return w.detach(), x.grad
    return _conv64(case, seed, d, row, col, n)


def _conv64(case, seed, d, row, col, n):
    """The layer in 64 bits: per-edge messages of the tensor-product paths, summed over targets."""
    conv = _layer(case, seed).double()
    u, dist, y = _geometry(d["pos"], row, col)
    u, dist, y = u.float().double(), dist.float().double(), y.float().double()  # as a program holds them
    train = case["train"]
    feats = [d[x].double().requires_grad_(train) if d[x] is not None else None for x in ("s", "v", "t")]
    rb = conv.radial_basis

    def mix(w, x):
        return (x.transpose(1, 2) @ w.weight.t()).transpose(1, 2)

    with torch.set_grad_enabled(train):
        basis = torch.sin(rb.freqs * dist[:, None]) / dist.clamp(min=1e-8)[:, None]
        env = (0.5 * (1 + torch.cos(math.pi * dist / rb.cutoff))).clamp(min=0)
        R = rb.mlp(basis * env[:, None])
        s, v = feats[0][row], feats[1][row]
        t = feats[2][row] if feats[2] is not None else None
        y0, c = y[:, :1], iter(range(9))
        r = [R[:, i:i + 1] for i in range(R.shape[1])]
        ms = r[next(c)] * y0 * (s @ conv.w_ss.weight.t())
        mv = (r[next(c)] * (s @ conv.w_sv.weight.t()))[..., None] * u[:, None]
        mv = mv + (r[next(c)] * y0)[..., None] * mix(conv.w_vv_scalar, v)
        ms = ms + r[next(c)] * ((v * u[:, None]).sum(-1) @ conv.w_vs.weight.t())
        cross = torch.linalg.cross(u[:, None].expand_as(v), v, dim=-1)
        mv = mv + r[next(c)][..., None] * mix(conv.w_vv_cross, cross)
        avg = _average_degree(row, col, n, case["b"])
        mt = None
        if t is not None:
            y2 = y[:, 4:9]
            mt = (r[next(c)] * (s @ conv.w_st2.weight.t()))[..., None] * y2[:, None]
            mt = mt + (r[next(c)] * y0)[..., None] * mix(conv.w_t2t2, t)
            outer = (u[:, None, :, None] * v[:, :, None, :]).flatten(2)
            mt = mt + r[next(c)][..., None] * mix(conv.w_vt2, outer @ conv.cg_11_2.reshape(9, 5))
            ms = ms + r[next(c)] * ((t * t).sum(-1) @ conv.w_t2s.weight.t())

        def collect(m):
            z = torch.zeros((n,) + m.shape[1:], dtype=torch.float64, device=DEV).index_add(0, col, m)
            return z / avg.reshape((n,) + (1,) * (m.dim() - 1))

        outs = [collect(ms) + conv.scalar_bias, collect(mv)] + ([collect(mt)] if mt is not None else [])
        if not train:
            return tuple(outs)
        torch.autograd.backward(outs, [d[x].double() for x in ("gs", "gv", "gt") if d[x] is not None])
    return dict(out=[x.detach() for x in outs], feat=[x.grad for x in feats if x is not None],
                weight=[p.grad for p in conv.parameters()])
