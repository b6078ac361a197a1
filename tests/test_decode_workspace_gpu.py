"""Decode attention with workspaces of every small context: the parts a row may be cut into follow the workspace's slots."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ctx", [[1], [64], [65, 3], [128], [900], [1030, 64, 1], [2000] * 5, [1100, 17, 300] * 12])
@pytest.mark.parametrize("spare", [0, 5000])
def test_decode_with_a_tight_workspace(ctx, spare):
    from financial_chatbot_llm_amd import ops
    g = torch.Generator(device="cuda").manual_seed(sum(ctx))
    B, Hq, Hkv, D = len(ctx), 8, 2, 128
    nb = [-(-c // 64) for c in ctx]
    kc, vc = (torch.zeros(sum(nb), Hkv, 64 * D, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    bt = torch.zeros(B, max(nb), dtype=torch.int32)
    rows, at = [], 0
    for i, n in enumerate(nb):
        bt[i, :n] = torch.arange(at, at + n)
        kv = torch.randn(n * 64, 2 * Hkv * D, generator=g, device="cuda").to(torch.bfloat16)
        rows.append(kv)
        slots = torch.arange(at * 64, (at + n) * 64, dtype=torch.int32, device="cuda")
        ops.rope_kv_write(torch.cat([kv.new_zeros(n * 64, Hq * D), kv], 1), slots, None, slots, kc, vc, Hq, Hkv, D, apply_rope=False)
        at += n
    q = torch.randn(B, Hq, D, generator=g, device="cuda").to(torch.bfloat16)
    ws = ops.DecodeWorkspace.create(B, Hq, D, max(ctx) + spare, "cuda")
    got = ops.decode(q, torch.tensor(ctx, dtype=torch.int32, device="cuda"), bt.cuda(), kc, vc, D ** -0.5, workspace=ws).float()
    for i, c in enumerate(ctx):
        k, v = rows[i][:c].float().view(c, 2, Hkv, D).unbind(1)
        k, v = (t.permute(1, 0, 2).repeat_interleave(Hq // Hkv, 0).contiguous() for t in (k, v))
        p = torch.softmax((k * q[i].float()[:, None]).sum(-1) * D ** -0.5, -1)
        want = (p[:, :, None] * v).sum(1)
        assert float((got[i] - want).norm() / want.norm()) < 8e-3       # weights and output in bf16
