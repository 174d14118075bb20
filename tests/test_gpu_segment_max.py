"""Segment max where its kernels branch: steps with and without NaNs in one segment, signed zeros,
infinities, ties, merged and whole-wave forwards, and the backward's record and message reads; the
bfloat16 mean backward on both sides of its reciprocal rule.  Bit-exact against the oracle."""

import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu


def _np(t):
    return t.float().cpu().numpy() if t.dtype == torch.bfloat16 else t.cpu().numpy()


def _csr(S, deg, g, shuffled):
    d = torch.randint(0, deg + 1, (S,), generator=g)
    col = torch.repeat_interleave(torch.arange(S), d)
    if shuffled:
        col = col[torch.randperm(col.numel(), generator=g)]
    col[::53] = S + 1  # rows of no segment
    return col


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float64])
@pytest.mark.parametrize("S, deg, C", [(4096, 9, 64), (4096, 40, 8), (5000, 3, 33), (4100, 17, 130),
                                       (300, 200, 64), (7, 900, 5)])
@pytest.mark.parametrize("special", [False, True])
def test_segment_max(dev, S, deg, C, dtype, special):
    from gdl_amd.csrc import (segment_reduce_backward_hip, segment_reduce_forward_hip,
                              sort_and_build_csr_cuda)
    g = torch.Generator().manual_seed(S + deg + C)
    col = _csr(S, deg, g, special)
    E = col.numel()
    msg = torch.randn(E, C, generator=g)
    if special:
        msg = (msg * 2).round() / 2                     # ties, and zeros of both signs
        pick = torch.rand(E, C, generator=g)
        msg[pick < 0.01] = float("nan")
        msg[(pick > 0.5) & (pick < 0.55)] = -float("inf")
        msg[pick > 0.995] = float("inf")
    msg = msg.to(dtype)
    cs, pm, ns, ne = sort_and_build_csr_cuda(col.to(dev), S)
    for ties in (0, 1):
        out, arg = segment_reduce_forward_hip(msg.to(dev), pm, ns, ne, S, "max", ties)
        want, warg = oracle.segment_reduce_fwd(_np(msg), pm.cpu().numpy(), ns.cpu().numpy(),
                                               ne.cpu().numpy(), S, "max", ties)
        np.testing.assert_array_equal(arg.cpu().numpy(), warg)
        np.testing.assert_array_equal(_np(out).astype(np.float64), want)
        assert np.array_equal(np.signbit(_np(out))[want == 0], np.signbit(want)[want == 0])
        grad = torch.randn(S, C, generator=g).to(dtype)
        got = segment_reduce_backward_hip(grad.to(dev), cs, pm, ns, ne, E, "max", msg=msg.to(dev),
                                          out=out, arg=arg)
        ref = oracle.segment_reduce_bwd(_np(grad), cs.cpu().numpy(), pm.cpu().numpy(), ns.cpu().numpy(),
                                        ne.cpu().numpy(), E, "max", msg=_np(msg), out=want, arg=warg,
                                        dtype=str(dtype).split(".")[-1])
        np.testing.assert_array_equal(_np(got).astype(np.float64), ref)


def test_segment_max_backward_without_segments(dev):
    """No segment: every row is zero (through the C entry point, which takes S = 0)."""
    from gdl_amd import _native as nat
    cs = torch.zeros(9, dtype=torch.int32, device=dev)
    msg = torch.ones(9, 4, device=dev)
    arg = torch.zeros(1, 4, dtype=torch.int32, device=dev)
    got = torch.full((9, 4), float("nan"), device=dev)
    nat.check(nat.lib().geo_segment_reduce_bwd(
        nat.REDUCE_CODES["max"], nat.DTYPE_CODES[msg.dtype], nat.ptr(msg), nat.ptr(msg), nat.ptr(msg),
        nat.ptr(arg), nat.ptr(cs), None, nat.ptr(cs), nat.ptr(cs), 9, 0, 4, nat.ptr(got),
        nat.stream_of(torch.device(dev))), "geo_segment_reduce_bwd")
    assert torch.equal(got, torch.zeros_like(got))


@pytest.mark.parametrize("sizes", [[3, 1, 0, 7, 4095, 4096], [4097, 5], [6000, 4096, 2]])
def test_bfloat16_mean_backward_rounds_the_quotient(dev, sizes):
    from gdl_amd.csrc import segment_reduce_backward_hip, sort_and_build_csr_cuda
    S = len(sizes)
    col = torch.repeat_interleave(torch.arange(S), torch.tensor(sizes))
    cs, pm, ns, ne = sort_and_build_csr_cuda(col.to(dev), S)
    bits = torch.arange(0, 0x7f81, 13, dtype=torch.int32)  # all magnitudes, infinity at the end
    grad = bits.to(torch.int16).view(torch.bfloat16)[:2504].reshape(1, -1).repeat(S, 1).contiguous()
    got = segment_reduce_backward_hip(grad.to(dev), cs, pm, ns, ne, col.numel(), "mean").cpu()
    want = (grad.float() / torch.tensor(sizes).clamp(min=1).float()[:, None]).bfloat16()[col]
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
