"""Sublayer outputs that the norm behind them adds up (slices of K, routed rows, a shared expert) against the same outputs written out
first: the sums and roundings are the same ones in the same order, so the results are equal bit for bit."""
import pytest
import torch

from financial_chatbot_llm_amd.ops import mixers as mx
from financial_chatbot_llm_amd.ops.gemm import Slabs

pytestmark = pytest.mark.gpu

DTS = [torch.float32, torch.bfloat16]


def randn(g, *s, dt=torch.float32):
    return torch.randn(*s, generator=g).to("cuda", dt)


def plain(g, T, W, dt, pad=0, off=0):
    return randn(g, T, W + pad, dt=dt)[:, off:off + W]


def slabs(g, S, T, W, dt):
    return Slabs(randn(g, S, T, W), dt)


def routed(g, T, W, dt, E=5, identity=2, top=3, shared=None, wts=True, pad=0):
    idx = torch.stack([torch.randperm(E + identity, generator=g)[:top] for _ in range(T)]).to(torch.int32).cuda()
    pos = torch.randperm(T * top, generator=g).view(T, top).to(torch.int32).cuda()
    w = randn(g, T, top) if wts else None
    if wts:
        w[0, 0] = 0.0                      # an entry of weight 0 is not read: its row may hold anything
    ys, h = plain(g, T * top, W, dt, pad), plain(g, T, W, dt, pad)
    if wts and int(idx[0, 0]) < E:
        ys[int(pos[0, 0])] = float("nan")
    return mx.Routed(ys, pos, idx, w, h, shared, E, identity > 0)


def outputs(g, T, W, dt):
    yield slabs(g, 2, T, W, dt)
    yield slabs(g, 8, T, W, dt)
    yield routed(g, T, W, dt)
    yield routed(g, T, W, dt, shared=plain(g, T, W, dt, 8, 4), top=4, pad=4)
    yield routed(g, T, W, dt, shared=slabs(g, 4, T, W, dt), top=1)
    yield routed(g, T, W, dt, identity=0, top=5, wts=False)
    yield routed(g, T, W, dt, pad=1)                 # rows off whole fours: written out first


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("T,W", [(1, 4), (3, 260), (2, 2052), (5, 4096), (2, 8192), (2, 8196), (3, 6)])
def test_parts_are_added_as_written_out(dt, T, W):
    g = torch.Generator().manual_seed(W + T)
    w, wa, wb = randn(g, W), randn(g, W), randn(g, W)
    n1, n2 = mx.DynTanh(0.7, randn(g, W), randn(g, W)), mx.DynTanh(0.4, randn(g, W), randn(g, W))
    other = plain(g, T, W, dt)
    for v in outputs(g, T, W, dt):
        if isinstance(v, Slabs) and W % 8:
            continue                                  # products have columns in sixteens
        if isinstance(v, mx.Routed) and isinstance(v.shared, Slabs) and W % 8:
            v = v._replace(shared=None)
        x0 = randn(g, T, W)
        for fn in (lambda x, a: mx.residual_norm(x, w, 1e-5, a, out_dtype=dt),
                   lambda x, a: mx.residual_norm(x, w, 1e-5, a, other, 0.5, dt, 0.3),
                   lambda x, a: mx.residual_norm(x, w, 1e-5, other, a, 0.5, dt),
                   lambda x, a: mx.post_norm_add(x, a, w, 1e-5, dt),
                   lambda x, a: mx.post_norm_add(x, other, w, 1e-5, dt, a, wa, wb),
                   lambda x, a: mx.dyn_tanh_residual(x, a, n1, n2, dt),
                   lambda x, a: mx.dyn_tanh_residual(x, a, n1)):
            xp, xw = x0.clone(), x0.clone()
            got, want = fn(xp, v), fn(xw, v.materialize())
            assert torch.equal(xp, xw) and bool(torch.isfinite(xp).all())
            assert (got is None and want is None) or torch.equal(got, want)


@pytest.mark.parametrize("dt", DTS)
def test_routed_rows_of_the_written_stream(dt):
    """The stream itself as the routed input (f32 decoders): identity rows are read before the update."""
    g = torch.Generator().manual_seed(1)
    T, W = 4, 512
    for identity in (0, 2):
        x0, w = randn(g, T, W), randn(g, W)
        r = routed(g, T, W, torch.float32, identity=identity)
        xp, xw = x0.clone(), x0.clone()
        got = mx.residual_norm(xp, w, 1e-5, r._replace(h=xp), out_dtype=dt)
        want = mx.residual_norm(xw, w, 1e-5, r._replace(h=xw).materialize(), out_dtype=dt)
        assert torch.equal(xp, xw) and torch.equal(got, want)
