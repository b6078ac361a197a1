"""The second factors of low-rank projections (``mx_low_rank``) against float64: ranks, widths around a wave's and a block's columns, rows
around a tile and a block's walk, columns of a wider projection, values that are not finite, and the layouts that keep the products."""
import pytest
import torch

from financial_chatbot_llm_amd.ops import _native as N, mixers as mx

pytestmark = pytest.mark.gpu


def operands(dt, T, ra, na, rg, ng, pad=8, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed + T + na)
    rows = torch.randn((T, pad + ra + rg), generator=g, device="cuda").to(dt)
    wa = torch.randn((na, ra), generator=g, device="cuda") * ra ** -0.5
    wg = (torch.randn((ng, rg), generator=g, device="cuda") * max(rg, 1) ** -0.5).to(dt)
    return rows[:, pad:pad + ra], wa, rows[:, pad + ra:], wg


def check(a, g, ua, wa, ug, wg, dt):
    want = ua.double() @ wa.double().t()
    # K additions in f32, each rounded by up to 2^-24 of a sum that is at most that of the magnitudes
    f32 = lambda u, w: u.shape[1] * 2.0 ** -24 * (u.double().abs() @ w.double().abs().t())  # noqa: E731
    assert a.dtype == torch.float32 and ((a.double() - want).abs() <= f32(ua, wa)).all()
    if wg is not None:
        want = ug.double() @ wg.double().t()
        e = 2.0 ** -8 if dt == torch.bfloat16 else 0.0
        assert g.dtype == dt and ((g.double() - want).abs() <= e * want.abs() + f32(ug, wg)).all()


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T", [1, 15, 16, 17, 130, 3453])
@pytest.mark.parametrize("ra,na,rg,ng", [(64, 2048, 64, 2048), (32, 1024, 0, 0), (64, 16, 32, 272), (32, 80, 64, 64)])
def test_against_float64(dt, T, ra, na, rg, ng, monkeypatch):
    ua, wa, ug, wg = operands(dt, T, ra, na, rg, ng)
    ug, wg = (ug, wg) if ng else (None, None)
    calls, mcall = [], N.mcall
    monkeypatch.setattr(N, "mcall", lambda name, *a: (calls.append(name), mcall(name, *a))[1])
    a, g = mx.low_rank(ua, wa, ug, wg)
    assert calls == ["mx_low_rank"]
    check(a, g, ua, wa, ug, wg, dt)


@pytest.mark.parametrize("K", [32, 64])
@pytest.mark.parametrize("spread", [0.0, 2.0])
def test_no_less_exact_than_the_f32_product(K, spread):
    """The sums over exact pieces of the weights against those of the product that they stand for, on f32 rows of the same values: weights of one size,
    and spread over some orders of magnitude."""
    ua, wa, _, _ = operands(torch.bfloat16, 1500, K, 2048, 0, 0, seed=K)
    g = torch.Generator(device="cuda").manual_seed(K)
    wa = wa * torch.exp(spread * torch.randn(wa.shape, generator=g, device="cuda"))
    want, size = ua.double() @ wa.double().t(), ua.double().abs() @ wa.double().abs().t()
    here, before = ((y.double() - want).abs() for y in (mx.low_rank(ua, wa)[0], torch.nn.functional.linear(ua.float(), wa)))
    assert here.norm() <= before.norm()
    # three products for each 32 of K, each of which adds 32 terms to the sum: K / 32 * 3 roundings of at most 2^-24 of the magnitudes, and as much again
    # for what the unit cuts while it aligns a product's terms
    assert (here <= K / 32 * 6 * 2.0 ** -24 * size).all(), float((here / size).max() * 2 ** 24)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_values_that_are_not_finite(dt):
    ua, wa, ug, wg = operands(dt, 40, 64, 96, 64, 96)
    wa[5, 3], wa[6, 0], wa[7, 1], ua[18, 4], ua[33, 9] = float("inf"), float("-inf"), float("nan"), float("inf"), float("nan")
    wa[:, 4] = torch.where(wa[:, 4] > 0, 1.0, -1.0)           # weights of one piece: the others are zeros beside the infinity
    a, _ = mx.low_rank(ua, wa, ug, wg)
    want = ua.double() @ wa.double().t()
    assert torch.equal(a.isnan(), want.isnan()) and torch.equal(a.isinf(), want.isinf())
    assert torch.equal(a[want.isinf()].double(), want[want.isinf()])
    ok = want.isfinite()
    assert ((a.double() - want).abs()[ok] <= 1e-4).all()


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("ra,na,rg,ng,pad", [(48, 64, 48, 64, 8), (64, 72, 64, 64, 8), (64, 64, 64, 64, 3), (64, 64, 16, 64, 8)])
def test_other_layouts_keep_the_products(dt, ra, na, rg, ng, pad):
    ua, wa, ug, wg = operands(dt, 20, ra, na, rg, ng, pad)
    a, g = mx.low_rank(ua, wa, ug, wg)
    check(a, g, ua, wa, ug, wg, dt)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_autocast_and_gradients(dt):
    """As the two products: autocast's type, and gradients for rows and weights."""
    ua, wa, ug, wg = operands(dt, 20, 64, 64, 32, 80)
    with torch.autocast("cuda", dtype=torch.float16):
        a, g = mx.low_rank(ua, wa, ug, wg)
        want = torch.nn.functional.linear(ua.float(), wa), torch.nn.functional.linear(ug, wg)
    assert a.dtype == g.dtype == torch.float16 and torch.equal(a, want[0]) and torch.equal(g, want[1])
    for i in range(4):
        ts = [t.detach().clone() for t in (ua, wa, ug, wg)]
        ts[i].requires_grad_()
        a, g = mx.low_rank(*ts)
        (a if i < 2 else g).sum().backward()
        u, w = ts[:2] if i < 2 else ts[2:]
        want = (w if i % 2 == 0 else u).double().sum(0)
        # sums of at most 80 products with ones: f32, and in bf16 the result rounded to eight significant bits
        e = 2.0 ** -8 if ts[i].dtype == torch.bfloat16 else 0.0
        size = (w if i % 2 == 0 else u).double().abs().sum(0)
        assert ((ts[i].grad.double() - want).abs() <= e * want.abs() + 80 * 2.0 ** -24 * size).all()
    assert not any(t.requires_grad for t in mx.low_rank(ua, wa, ug, wg))


@pytest.mark.parametrize("T,here", [(128 * 65535, True), (128 * 65535 + 1, False), (1 << 23, False)])
def test_most_rows(T, here, monkeypatch):
    """The launch has a block of its grid for each 128 rows; more rows are the product's."""
    ua = torch.ones((T, 32), dtype=torch.bfloat16, device="cuda")
    ua[-1] = 2.0
    calls, mcall = [], N.mcall
    monkeypatch.setattr(N, "mcall", lambda name, *a: (calls.append(name), mcall(name, *a))[1])
    a, _ = mx.low_rank(ua, torch.ones((16, 32), device="cuda"))
    assert bool(calls) is here and (a[:-1] == 32.0).all() and (a[-1] == 64.0).all()
