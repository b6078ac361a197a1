"""A matrix per head on strided rows of heads (``ops.mixers.HeadLinear``) against float64: both kernel forms, edges of the token
tiles, odd numbers of column groups, views off the kernel's 16 bytes, and the sizes that keep the batched product."""
import pytest
import torch

from financial_chatbot_llm_amd.ops import mixers as mx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T", [1, 2, 15, 17, 64, 512, 513, 1000])
@pytest.mark.parametrize("H,N,K", [(16, 256, 96), (3, 96, 256), (1, 16, 32), (2, 48, 64), (5, 40, 24), (2, 512, 160)])
def test_against_float64(dt, T, H, N, K):
    g = torch.Generator().manual_seed(T + N)
    w = (torch.randn((H, N, K), generator=g) * K ** -0.5).to(dt).cuda()
    q = torch.randn((T, H * (K + 32) + 8), generator=g).to(dt).cuda()
    f = mx.HeadLinear(w)
    assert f.native == (N % 16 == 0 and K % 32 == 0)
    for off in (0, 8, 3):                                    # 3: rows off the kernel's 16 bytes
        x = q[:, off:off + H * (K + 32)].unflatten(1, (H, K + 32))[:, :, :K]
        y = f(x)
        want = torch.einsum("thk,hnk->thn", x.double().cpu(), w.double().cpu())
        assert y.is_contiguous() and y.shape == (T, H, N)
        # one rounding of the result to eight significant bits (half a unit: 2^-8 of it at most); sums of K f32 products
        e = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -20
        assert ((y.double().cpu() - want).abs() <= want.abs() * e + 2.0 ** -18 * K ** 0.5).all()


def test_weights_off_16_bytes():
    """A part of a flat buffer of weights, as a loader may hand it over."""
    w, x = torch.randn(3 * 32 * 64 + 3, device="cuda")[3:].view(3, 32, 64), torch.randn((5, 3, 64), device="cuda")
    assert ((mx.HeadLinear(w)(x).double() - (x.double()[:, :, None] * w.double()).sum(-1)).abs() <= 2.0 ** -18 * 64).all()


@pytest.mark.parametrize("dt,T,H,N,K,native", [
    (torch.bfloat16, 8192, 32, 128, 256, True), (torch.bfloat16, 8193, 32, 128, 256, False), (torch.float32, 1024, 32, 128, 256, True),
    (torch.float32, 1025, 32, 128, 256, False), (torch.float32, 1025, 32, 256, 128, True), (torch.bfloat16, 3, 2, 512, 96, False),
    (torch.bfloat16, 3, 2, 256, 128, True), (torch.bfloat16, 3, 2, 256, 160, False)])
def test_rule(dt, T, H, N, K, native, monkeypatch):
    """Large matrices, and a long K beside many rows, keep the batched product."""
    from financial_chatbot_llm_amd.ops import _native as nat
    calls = []
    mcall = nat.mcall
    monkeypatch.setattr(nat, "mcall", lambda name, *a: (calls.append(name), mcall(name, *a))[1])
    g = torch.Generator(device="cuda").manual_seed(T)
    w = torch.randn((H, N, K), generator=g, device="cuda").mul_(K ** -0.5).to(dt)
    x = torch.randn((T, H, K), generator=g, device="cuda").to(dt)
    y = mx.HeadLinear(w)(x)
    assert calls == (["mx_head_linear"] if native else [])
    want = (x[:50].double()[:, :, None] * w.double()).sum(-1)
    e = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -20
    assert ((y[:50].double() - want).abs() <= want.abs() * e + 2.0 ** -18 * K ** 0.5).all()
