"""The grouped fp8 products of a decode step: experts with pairs around every token tile and chunk, both widths of workgroup, K around the
numbers of waves that split it and of k-pairs in flight."""
import pytest
import torch

from financial_chatbot_llm_amd.ops import _native as N
from financial_chatbot_llm_amd.ops import moe

pytestmark = pytest.mark.gpu

COUNTS = [1, 0, 16, 17, 33, 48, 65, 130]


@pytest.mark.parametrize("ntf", [2, 4])
@pytest.mark.parametrize("epi", [1, 2])
@pytest.mark.parametrize("K", [64, 192, 256, 512, 1536, 2048, 8192, 8448])
def test_pairs_by_expert(K, epi, ntf):
    g = torch.Generator().manual_seed(K + epi)
    E, n, P, T = len(COUNTS), 128, sum(COUNTS), 70
    w8, s = moe.quantize_fp8_rowwise(torch.randn(E, n, K, generator=g) * K ** -0.5)
    x8 = torch.randn(T, K, generator=g).to(torch.float8_e4m3fn)
    xs, rw = torch.rand(T, generator=g) + 0.5, torch.rand(P, generator=g)
    rows = torch.randint(0, T, (P,), generator=g).int()
    off = torch.tensor([0] + COUNTS).cumsum(0).int()
    xq, xsc = (x8, xs) if epi == 1 else (x8[rows.long()], xs[rows.long()])
    y = torch.zeros(P, n // 2 if epi == 1 else n, dtype=torch.bfloat16, device="cuda")
    d = [t.cuda().contiguous() for t in (xq.view(torch.uint8), xsc, rows, off, s, rw)]
    wt = moe.tile_fp8_weight(w8.cuda())
    N.call("penny_moe_gemm_fp8", N.ptr(d[0]), N.ptr(d[1]), N.ptr(d[2]) if epi == 1 else None, N.ptr(d[3]), N.ptr(wt), N.ptr(d[4]),
           N.ptr(d[5]), N.ptr(y), E, n, K, epi, ntf, N.stream())
    expert = torch.repeat_interleave(torch.arange(E), torch.tensor(COUNTS))
    W = w8.view(torch.float8_e4m3fn).double() if w8.dtype == torch.uint8 else w8.double()
    W, X = W * s.double()[..., None], x8.double() * xs.double()[:, None]
    W, X = W.cuda(), X.cuda()[rows.long()]
    full, size = (torch.stack([W_[e] @ X_ for e, X_ in zip(expert.tolist(), X_all)]) for W_, X_all in ((W, X), (W.abs(), X.abs())))
    # f32 sums of what the matrix unit gives for 32 fp8 products (aligned to the largest, low bits cut: 2^-17.6 of their sizes was met at
    # K = 64, where nothing else is added); one rounding to bf16 is 2^-8 of the value at most
    slack = (K * 2.0 ** -24 + 2.0 ** -17) * size + 1e-30
    if epi == 2:
        ref, tol = full * d[5].double()[:, None], (slack + 2.0 ** -8 * full.abs()) * d[5].double()[:, None] * 1.01
    else:
        def half(a, i):
            return a.view(P, n // 32, 2, 16)[:, :, i].reshape(P, n // 2)
        G, U, e = half(full, 0), half(full, 1), 2.0 ** -8
        act = G * torch.sigmoid(G)
        ref = act * U                                         # the gate's slope is at most 1.1; gate, up, activation and result rounded
        tol = 1.05 * (U.abs() * (1.1 * (G.abs() * e + half(slack, 0)) + e * act.abs()) + act.abs() * (2 * e * U.abs() + half(slack, 1))) + 1e-30
    err = (y.double() - ref).abs()
    assert bool((err <= tol).all()), float((err / tol).max())


@pytest.mark.parametrize("K", [256, 1536, 4096, 14336])
def test_widths_agree(K):
    """One token's row of an expert in a small batch and in a large one, whose products split K over other numbers of waves."""
    g = torch.Generator().manual_seed(K)
    n, P = 128, 40
    w8, s = moe.quantize_fp8_rowwise(torch.randn(1, n, K, generator=g) * K ** -0.5)
    x8 = torch.randn(P, K, generator=g).to(torch.float8_e4m3fn)
    xs, rw = torch.rand(P, generator=g) + 0.5, torch.ones(P)
    wt, d = moe.tile_fp8_weight(w8.cuda()), [t.cuda().contiguous() for t in (x8.view(torch.uint8), xs, s, rw)]

    def rows(first, count, ntf):
        y = torch.zeros(count, n, dtype=torch.bfloat16, device="cuda")
        off = torch.tensor([0, count], dtype=torch.int32, device="cuda")
        N.call("penny_moe_gemm_fp8", N.ptr(d[0][first:]), N.ptr(d[1][first:]), None, N.ptr(off), N.ptr(wt), N.ptr(d[2]), N.ptr(d[3][first:]), N.ptr(y),
               1, n, K, 2, ntf, N.stream())
        return y.double()
    thin, wide = rows(7, 1, 2), rows(0, P, 4)[7:8]
    W = w8.view(torch.float8_e4m3fn).double().cuda()[0] * s.double().cuda()[0][:, None]
    size = (x8.double().cuda()[7:8] * xs.double().cuda()[7]).abs() @ W.abs().t()
    # either sum is within K 2^-24 of the magnitudes and the matrix unit's own cut (above), and is rounded to bf16
    assert ((thin - wide).abs() <= 2 * (K * 2.0 ** -24 + 2.0 ** -17) * size + 2.0 ** -7 * wide.abs()).all()
    assert torch.equal(rows(7, 1, 4), wide)                    # of one width, whatever the batch: the same bits


def test_row_groups():
    assert moe.moe_ntf(96, 8, 28672, 4096) == (2, 4) and moe.moe_ntf(320, 8, 28672, 4096) == (4, 4)
    assert moe.moe_ntf(159, 8, 28672, 2048) == (2, 2) and moe.moe_ntf(160, 8, 28672, 2048) == (4, 4)
    assert moe.moe_ntf(2, 8, 28672, 4096) == (2, 2) and moe.moe_ntf(16, 8, 28688, 4080) == (4, 4)
