"""Matrix-state scans in chunks of 16 tokens (gla and delta): segment lengths around the chunk, key and value sizes around the
tiles, strong and weak decays, against the token recurrence in 64 bits; and a value that is not finite reaches no earlier
token."""
import pytest
import torch
import torch.nn.functional as F

from financial_chatbot_llm_amd.ops import mixers as mx

pytestmark = pytest.mark.gpu

LENS = [70, 33, 16, 1, 0, 47, 32]


def inputs(H, G, D, P, dt, shift, seed=3):
    g = torch.Generator().manual_seed(seed)
    T = sum(LENS) + 3                                                # rows behind the last segment belong to nobody
    r = lambda *s: torch.randn(s, generator=g)
    x = {"q": r(T, G * D + 8).to(dt), "k": r(T, G * D).to(dt), "v": r(T, H * P + 4).to(dt), "a": r(T, H * D) + shift,
         "a_bias": r(H * D) * 0.1, "A_log": r(H) * 0.5, "beta": r(T, H).to(dt), "state": r(len(LENS) + 1, H, D, P)}
    x["cu"] = torch.tensor([0] + torch.tensor(LENS).cumsum(0).tolist(), dtype=torch.int32)
    x["slot"] = torch.tensor([5, 0, 7, -1, 2, 3, 6], dtype=torch.int32)   # the fourth is padding
    pos = [torch.arange(n) + (7 if i % 2 else 0) for i, n in enumerate(LENS)]
    x["pos"] = torch.cat(pos + [torch.zeros(3, dtype=torch.int64)]).int()
    return x


def run(x, H, G, D, P, mode):
    y = {k: t.cuda() for k, t in x.items()}
    o = mx.matrix_scan(y["q"][:, :G * D], y["k"], y["v"][:, :H * P], y["a"], y["a_bias"], y["state"], y["cu"], y["slot"],
                       y["pos"], H, G, D, P, mode, tau=16.0, A_log=y["A_log"], beta=y["beta"], max_len=max(LENS))
    return o.cpu(), y["state"].cpu()


def exact(x, H, G, D, P, mode):
    y = {k: t.double() if t.is_floating_point() else t for k, t in x.items()}
    T = y["q"].shape[0]
    q, k, v = y["q"][:, :G * D].view(T, G, D), y["k"].view(T, G, D), y["v"][:, :H * P].view(T, H, P)
    z = (y["a"] + y["a_bias"]).view(T, H, D)
    if mode == "delta":
        q, k = (t * torch.rsqrt((t * t).sum(-1, keepdim=True) + 1e-6) for t in (q, k))
        dec, b = torch.exp(-torch.exp(y["A_log"])[:, None] * F.softplus(z)), torch.sigmoid(y["beta"])
    else:
        dec = torch.exp(-F.softplus(-z) / 16.0)
    q, k = (q * D ** -0.5).repeat_interleave(H // G, 1), k.repeat_interleave(H // G, 1)
    out, size, state = torch.zeros(T, H, P).double(), torch.zeros(T, H, P).double(), y["state"].clone()
    for s, n in enumerate(LENS):
        r0, sl = int(x["cu"][s]), int(x["slot"][s])
        if n == 0 or sl < 0:
            continue
        S = state[sl] if x["pos"][r0] != 0 else torch.zeros(H, D, P).double()
        for t in range(r0, r0 + n):
            S = dec[t][:, :, None] * S
            u = v[t]
            if mode == "delta":
                u = b[t][:, None] * (u - torch.einsum("hdp,hd->hp", S, k[t]))
            S = S + k[t][:, :, None] * u[:, None]
            out[t] = torch.einsum("hdp,hd->hp", S, q[t])
            size[t] = torch.einsum("hdp,hd->hp", S.abs(), q[t].abs())
        state[sl] = S
    return out.view(T, -1), state, size.view(T, -1)


@pytest.mark.parametrize("mode", ["gla", "delta"])
@pytest.mark.parametrize("shift", [-4.0, 0.0, 6.0, 60.0])
@pytest.mark.parametrize("H,G,D,P,dt", [(4, 2, 64, 16, torch.float32), (2, 2, 40, 33, torch.bfloat16),
                                        (4, 4, 128, 48, torch.float32), (3, 1, 129, 7, torch.float32),
                                        (2, 1, 256, 64, torch.bfloat16)])
def test_chunks(mode, shift, H, G, D, P, dt):
    x = inputs(H, G, D, P, dt, shift)
    got, state = run(x, H, G, D, P, mode)
    want, wstate, size = exact(x, H, G, D, P, mode)
    live = torch.zeros(x["q"].shape[0], dtype=torch.bool)
    for s, n in enumerate(LENS):
        live[x["cu"][s]:x["cu"][s] + n] = x["slot"][s] >= 0
    # f32: each of <= 70 tokens rounds the state, its decay and its products a few times, at the size of the sums of moduli
    tol = 2.0 ** -24 * (8 * max(LENS)) * (1 + size) / 4
    assert ((got.double() - want).abs()[live] <= tol[live]).all()
    assert ((state.double() - wstate).abs() <= 2.0 ** -24 * 8 * max(LENS) * (1 + wstate.abs())).all()


@pytest.mark.parametrize("mode", ["gla", "delta"])
@pytest.mark.parametrize("where", ["v", "k"])
def test_not_finite(mode, where):
    H, G, D, P = 2, 2, 64, 32
    x = inputs(H, G, D, P, torch.float32, 0.0)
    bad = int(x["cu"][0]) + 21
    clean, cstate = run({k: t.clone() for k, t in x.items()}, H, G, D, P, mode)
    x[where][bad, 5] = float("inf")
    got, state = run(x, H, G, D, P, mode)
    n = LENS[0]
    assert torch.equal(got[:bad], clean[:bad]) and torch.equal(got[n:n + 33], clean[n:n + 33])
    col = got.view(-1, H, P)[bad:n, 0, 5]
    assert not torch.isfinite(col).any() and not torch.isfinite(state[5, 0, :, 5]).all()
    if where == "v":                                                  # only that value column
        assert torch.equal(got.view(-1, H, P)[:n, 0, 6], clean.view(-1, H, P)[:n, 0, 6])


@pytest.mark.parametrize("mode", ["gla", "delta"])
@pytest.mark.parametrize("lens", [[1] * 30 + [33, 2, 0, 17] + [1] * 20, [32] + [1] * 7, [31, 32, 1, 1, 2, 3, 0, 1, 1], [70] * 7 + [1],
                                  [40] * 3 + [1] * 4, [32] * 8])
@pytest.mark.parametrize("D,P,dt", [(64, 16, torch.bfloat16), (128, 48, torch.float32), (256, 20, torch.bfloat16)])
def test_single_rows_beside_chunks(mode, lens, D, P, dt):
    """Steps short on average give their single rows to the single-row form, others take them along."""
    g = torch.Generator().manual_seed(len(lens) + D)
    H, G, T, S = 4, 2, sum(lens) + 2, len(lens)
    r = lambda *s: torch.randn(s, generator=g)  # noqa: E731
    x = [r(T, G * D).to(dt), r(T, G * D).to(dt), r(T, H * P).to(dt), r(T, H * D), r(H * D) * 0.1, r(S, H, D, P)]
    slot = torch.randperm(S, generator=g).int()
    slot[min(3, S - 1)] = -1                                          # padding
    meta = [torch.tensor([0] + lens).cumsum(0).int(), slot, torch.cat([torch.arange(n) + i % 2 for i, n in enumerate(lens + [2])]).int()]
    opt = {"A_log": r(H) * 0.5, "beta": r(T, H).to(dt)} if mode == "delta" else {"tau": 16.0}
    got = [t.cuda() for t in x]
    out = mx.matrix_scan(*got, *(t.cuda() for t in meta), H, G, D, P, mode, max_len=max(lens),
                         **{k: v.cuda() if torch.is_tensor(v) else v for k, v in opt.items()}).cpu()
    want = mx.matrix_scan(*x, *meta, H, G, D, P, mode, **opt)
    live = torch.cat([torch.full((n,), bool(slot[i] >= 0)) for i, n in enumerate(lens)] + [torch.zeros(2, dtype=torch.bool)])
    # f32 on both sides: each of <= 70 tokens rounds the state and its products a few times
    assert torch.allclose(out[live], want[live], rtol=1e-4, atol=2e-4) and torch.allclose(got[5].cpu(), x[5], rtol=1e-4, atol=2e-4)


@pytest.mark.parametrize("mode", ["gla", "delta"])
@pytest.mark.parametrize("D,H,P,lens", [(32, 16, 64, [40] * 16), (16, 32, 64, [70] * 16), (64, 32, 64, [65] * 16), (48, 16, 64, [33, 50] * 8),
                                        (96, 16, 64, [40] * 16), (32, 16, 64, [65] * 3)])
def test_many_chains(mode, D, H, P, lens):
    """Steps on both sides of the line from which small keys go token by token."""
    g = torch.Generator().manual_seed(D + len(lens))
    T, S = sum(lens), len(lens)
    r = lambda *s: torch.randn(s, generator=g)  # noqa: E731
    x = [r(T, H * D), r(T, H * D), r(T, H * P), r(T, H * D), r(H * D) * 0.1, r(S, H, D, P)]
    meta = [torch.tensor([0] + lens).cumsum(0).int(), torch.randperm(S, generator=g).int(),
            torch.cat([torch.arange(n) + i % 2 for i, n in enumerate(lens)]).int()]
    opt = {"A_log": r(H) * 0.5, "beta": r(T, H)} if mode == "delta" else {"tau": 16.0}
    got = [t.cuda() for t in x]
    out = mx.matrix_scan(*got, *(t.cuda() for t in meta), H, H, D, P, mode, max_len=max(lens),
                         **{k: v.cuda() if torch.is_tensor(v) else v for k, v in opt.items()}).cpu()
    want = mx.matrix_scan(*x, *meta, H, H, D, P, mode, **opt)
    # f32 on both sides: each of <= 70 tokens rounds the state and its products a few times
    assert torch.allclose(out, want, rtol=1e-4, atol=2e-4) and torch.allclose(got[5].cpu(), x[5], rtol=1e-4, atol=2e-4)
