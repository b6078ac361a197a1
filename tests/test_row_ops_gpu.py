"""Row kernels by fours (norms, squared ReLU, 4-tap convolution) against the CPU form, at sizes around a lane's, a wave's and
a block's share and in layouts that only the element-wise forms take (odd sizes, odd strides, odd offsets)."""
import pytest
import torch

from financial_chatbot_llm_amd.ops import mixers as mx

pytestmark = pytest.mark.gpu

DTS = [torch.float32, torch.bfloat16]


def rand(g, *s, dt=torch.float32):
    return torch.randn(*s, generator=g).to(dt)


def view(x, pad, off):
    """The same rows with a stride of pad more elements, off elements into the buffer."""
    b = torch.full((x.shape[0], x.shape[1] + pad), float("nan"), dtype=x.dtype, device="cuda")
    b[:, off:off + x.shape[1]] = x.cuda()
    return b[:, off:off + x.shape[1]]


def near(got, want, dt, scale=1.0):
    # f32: sums of up to 8192 squares in another order; bf16 results: one rounding on each side
    tol = (2e-6 if dt == torch.float32 else 2.0 ** -7) * scale
    err = (got.float().cpu() - want.float()).abs()
    assert bool((err <= tol * (1 + want.float().abs())).all()), float(err.max())


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("pad,off", [(0, 0), (8, 4), (3, 0), (4, 1)])
@pytest.mark.parametrize("groups,n", [(3, 4), (2, 64), (5, 68), (1, 128), (3, 256), (1, 260), (2, 512), (1, 1024), (1, 2052),
                                      (1, 8192), (1, 8196), (2, 65)])
def test_group_norm(dt, pad, off, groups, n):
    g = torch.Generator().manual_seed(n)
    x, z, w = rand(g, 5, groups * n), rand(g, 5, groups * n, dt=dt), rand(g, groups * n)
    for gate in (None, z):
        want = mx.group_norm(x, w, 1e-5, groups, gate=gate, out_dtype=dt)
        got = mx.group_norm(view(x, pad, off), w.cuda(), 1e-5, groups, gate=None if gate is None else view(gate, pad, off),
                            out_dtype=dt)
        near(got, want, dt)


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("pad,off", [(0, 0), (4, 4), (1, 0)])
@pytest.mark.parametrize("H,P", [(1, 4), (3, 64), (5, 100), (2, 128), (3, 256), (1, 257), (2, 260)])
def test_head_norm_gate(dt, pad, off, H, P):
    g = torch.Generator().manual_seed(P)
    o, z, w = rand(g, 7, H * P), rand(g, 7, H * P, dt=dt), rand(g, P)
    for act in ("silu", "sigmoid"):
        want = mx.head_norm_gate(o, w, 1e-5, z, H, act, dt)
        near(mx.head_norm_gate(view(o, pad, off), w.cuda(), 1e-5, view(z, pad, off), H, act, dt), want, dt)


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("pad,off", [(0, 0), (4, 4), (1, 0)])
@pytest.mark.parametrize("T,H,P", [(22000, 3, 4), (1400, 3, 64), (530, 5, 100), (1025, 2, 128), (342, 3, 256), (513, 2, 256)])
def test_head_norm_gate_of_many_heads(dt, pad, off, T, H, P):
    g = torch.Generator().manual_seed(P)
    o, z, w = rand(g, T, H * P), rand(g, T, H * P, dt=dt), rand(g, P)
    for act in ("silu", "sigmoid"):
        want = mx.head_norm_gate(o, w, 1e-5, z, H, act, dt)
        near(mx.head_norm_gate(view(o, pad, off), w.cuda(), 1e-5, view(z, pad, off), H, act, dt), want, dt)


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("pad", [0, 4, 1])
@pytest.mark.parametrize("W", [4, 1024, 1028, 2048, 4100, 8192, 8196, 777])
def test_post_norm(dt, pad, W):
    g = torch.Generator().manual_seed(W)
    x, a, b = rand(g, 3, W), rand(g, 3, W, dt=dt), rand(g, 3, W, dt=dt)
    wa, wb, w = rand(g, W), rand(g, W), rand(g, W)
    for two in (False, True):
        for given in (False, True) if not two else (True,):
            cx, dx = x.clone(), x.cuda()
            kw = dict(a=a if given else None, b=b if two else None, wa=wa if two else None, wb=wb if two else None)
            want = post(cx, w, dt, **kw)
            dev = {k: None if v is None else (view(v, pad, 0) if v.dim() == 2 else v.cuda()) for k, v in kw.items()}
            got = post(dx, w.cuda(), dt, **dev)
            near(got, want, dt, 2.0)
            near(dx, cx, torch.float32, 2.0)


def post(x, w, dt, a, b, wa, wb):
    return mx.layer_norm_out(x, w, 1e-5, dt) if a is None else mx.post_norm_add(x, a, w, 1e-5, dt, b, wa, wb)


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("pad,off", [(0, 0), (8, 8), (8, 4), (1, 1)])
@pytest.mark.parametrize("n", [4, 8, 2048, 2056, 100, 33])
def test_relu2(dt, pad, off, n):
    g = torch.Generator().manual_seed(n)
    x = rand(g, 5, n, dt=dt)
    x[0, 0], x[1, 1] = float("inf"), float("-inf")
    assert torch.equal(mx.relu2(view(x, pad, off)).cpu(), mx.relu2(x))


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("n", [120, 128, 252, 256])
def test_relu2_of_narrow_rows(dt, n):
    """On both sides of the widths from which rows go by 16 bytes."""
    x = rand(torch.Generator().manual_seed(n), 300, n, dt=dt)
    assert torch.equal(mx.relu2(x.cuda()).cpu(), mx.relu2(x))


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("pad", [0, 4, 1])
@pytest.mark.parametrize("C,K", [(4, 4), (1028, 4), (30, 4), (64, 3)])
def test_conv(dt, pad, C, K):
    g = torch.Generator().manual_seed(C + K)
    lens = [1, 3, 32, 33, 70, 8, 2]
    T = sum(lens)
    x, w, b, ib = rand(g, T, C, dt=dt), rand(g, C, K), rand(g, C), rand(g, C)
    state = rand(g, 8, K - 1, C)
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32)
    slot = torch.tensor([3, 0, 7, 2, 5, -1, 1], dtype=torch.int32)
    pos = torch.cat([torch.arange(n) + (9 if i % 2 else 0) for i, n in enumerate(lens)]).int()
    live = torch.cat([torch.full((n,), int(s) >= 0) for n, s in zip(lens, slot)])
    for act in ("silu", "none"):
        cs, ds = state.clone(), state.cuda()
        want = mx.conv_act(x, w, b, cs, cu, slot, pos, max(lens), act, in_bias=ib)
        got = mx.conv_act(view(x, pad, 0), w.cuda(), b.cuda(), ds, cu.cuda(), slot.cuda(), pos.cuda(), max(lens), act,
                          in_bias=ib.cuda())
        near(got[live.cuda()], want[live], torch.float32)
        near(ds, cs, torch.float32)


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("pad", [0, 4, 1])
@pytest.mark.parametrize("lens", [[900, 33, 70, 8, 2, 1, 100], [8] * 130])
def test_conv_by_four(dt, pad, lens):
    """Enough rows for the form by four channels, and layouts that it leaves to the other one."""
    C, K, T, S = 4612, 4, sum(lens), len(lens)
    g = torch.Generator().manual_seed(T)
    x, w, b, ib, state = rand(g, T, C, dt=dt), rand(g, C, K), rand(g, C), rand(g, C), rand(g, S + 1, K - 1, C)
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32)
    slot = torch.randperm(S + 1, generator=g)[:S].int()
    slot[3] = -1
    pos = torch.cat([torch.arange(n) + (9 if i % 2 else 0) for i, n in enumerate(lens)]).int()
    live = torch.cat([torch.full((n,), int(s) >= 0) for n, s in zip(lens, slot)])
    for act in ("silu", "none"):
        cs, ds = state.clone(), state.cuda()
        want = mx.conv_act(x, w, b, cs, cu, slot, pos, max(lens), act, in_bias=ib)
        got = mx.conv_act(view(x, pad, 0), w.cuda(), b.cuda(), ds, cu.cuda(), slot.cuda(), pos.cuda(), max(lens), act,
                          in_bias=ib.cuda())
        near(got[live.cuda()], want[live], torch.float32)
        near(ds, cs, torch.float32)
