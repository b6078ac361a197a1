"""The small launches of a decode step around their edges: split-K slabs added up inside the norm and the rotary pass (numbers of slabs
with a form of their own and the loop behind them, tokens where the workgroups change), and rows whose attention lies in few and many parts."""
import math

import pytest
import torch

from financial_chatbot_llm_amd import ops
from financial_chatbot_llm_amd.ops import _native as N
from test_kernels_gpu import _paged_setup, close, rnd

pytestmark = pytest.mark.gpu


def slabs(S, T, n):
    g = torch.Generator().manual_seed(100 * S + T)
    P = torch.randn(S, T, n, generator=g)
    x = P[0].clone()
    for s in range(1, S):
        x += P[s]                     # the kernels' order, so the same f32 sums
    return P.cuda(), x.to(torch.bfloat16).cuda()


@pytest.mark.parametrize("S", [1, 2, 3, 4, 5, 6, 7, 8, 9, 13])
@pytest.mark.parametrize("T,H", [(3, 4096), (65, 2048), (2, 16384), (1, 72)])
def test_norm_of_slabs(S, T, H):
    P, x = slabs(S, T, H)
    w, res = (1 + 0.1 * torch.randn(H)).to(torch.bfloat16).cuda(), torch.randn(T, H).to(torch.bfloat16).cuda()
    r, y = res.clone(), torch.empty_like(res)
    N.call("penny_rmsnorm_slabs", N.ptr(P), S, N.ptr(r), N.ptr(w), N.ptr(y), T, H, 1e-5, 1, N.stream())
    want = (x.float() + res.float()).to(torch.bfloat16)
    assert torch.equal(r, want)
    full = want.double()
    ref = full * (full.pow(2).mean(1, keepdim=True) + 1e-5).rsqrt() * w.double()
    # two roundings to bf16: 8 bits of significand, so at most 2^-8 of the value each
    assert bool(((y.double() - ref).abs() <= 2.0 ** -6.95 * ref.abs() + 1e-30).all())


@pytest.mark.parametrize("S,T", [(1, 1), (2, 64), (3, 65), (4, 128), (5, 129), (8, 2), (9, 5), (4, 513)])
@pytest.mark.parametrize("D,Hq,Hkv", [(128, 32, 8), (64, 6, 2), (128, 64, 64)])
def test_rotary_of_slabs(S, T, D, Hq, Hkv):
    P, x = slabs(S, T, (Hq + 2 * Hkv) * D)
    blocks = T // 64 + 2
    pos = (torch.arange(T, dtype=torch.int32) * 7 % 500).cuda()
    slot = torch.randperm(64 * blocks)[:T].int()
    slot[T // 2] = -1 if T > 2 else slot[T // 2]
    slot = slot.cuda()
    cs = ops.rope_cos_sin(D, 512, 10000.0).cuda()
    outs = []
    for slab in (True, False):
        q = torch.zeros(T, Hq, D, dtype=torch.bfloat16, device="cuda")
        k, v = (torch.zeros(blocks, Hkv, 64 * D, dtype=torch.bfloat16, device="cuda") for _ in "kv")
        rest = (N.ptr(pos), N.ptr(cs), N.ptr(slot), N.ptr(q), N.ptr(k), N.ptr(v), T, Hq, Hkv, D, 1, N.stream())
        if slab:
            N.call("penny_rope_kv_write_slabs", N.ptr(P), S, *rest)
        else:
            N.call("penny_rope_kv_write", N.ptr(x), *rest)
        outs.append((q, k, v))
    assert all(torch.equal(a, b) for a, b in zip(*outs))


@pytest.mark.parametrize("B", [1, 8])
def test_rows_in_parts(B, monkeypatch):
    monkeypatch.setattr(ops.attention, "LEAN_MIN_PER_WAVE", 1)
    g = torch.Generator().manual_seed(11)
    Hq, Hkv, D = 32, 8, 128
    ctxs = [64 * k - 3 for k in (3, 4, 5, 15, 16, 17, 33, 1)][:B] if B > 1 else [64 * 33]
    tables, kc, vc = _paged_setup(ctxs, Hkv, D, gen=g)
    q = rnd(len(ctxs), Hq, D, gen=g)
    ctx = torch.tensor(ctxs, dtype=torch.int32)
    ws = ops.DecodeWorkspace.create(len(ctxs), Hq, D, 64 * 8 * 40, "cuda")   # 40 slots a row
    out = ops.decode(q.cuda(), ctx.cuda(), tables.cuda(), kc.cuda(), vc.cuda(), 1 / math.sqrt(D), workspace=ws)
    close(out, ops.decode(q, ctx, tables, kc, vc, 1 / math.sqrt(D)), atol=2e-2)
