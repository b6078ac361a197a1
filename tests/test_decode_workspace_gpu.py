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


@pytest.mark.parametrize("ctx,least", [([900] * 4, 2), ([1800, 700, 900], 2), ([900] * 16, 4), ([1200] * 12, 4), ([400] * 32, 2),
                                       ([1200] * 24, 4), ([700, 1, 64, 65, 1536], 2), ([2000] * 5, 2)])
def test_plan_follows_the_contexts(ctx, least):
    """The served layout (table and workspace of the longest sequence a model takes) is walked like a tight one."""
    from financial_chatbot_llm_amd import ops
    from financial_chatbot_llm_amd.ops.attention import LEAN_META0
    g = torch.Generator(device="cuda").manual_seed(sum(ctx))
    B, Hq, Hkv, D = len(ctx), 32, 8, 128
    nb = [-(-c // 64) for c in ctx]
    kc, vc = (torch.randn(sum(nb), Hkv, 64 * D, generator=g, device="cuda").to(torch.bfloat16) for _ in range(2))
    q = torch.randn(B, Hq, D, generator=g, device="cuda").to(torch.bfloat16)
    lens = torch.tensor(ctx, dtype=torch.int32, device="cuda")
    got = []
    for width in (max(nb), 128):
        bt, at = torch.zeros(B, width, dtype=torch.int32), 0
        for i, n in enumerate(nb):
            bt[i, :n] = torch.arange(at, at + n)
            at += n
        ws = ops.DecodeWorkspace.create(B if width < 128 else 64, Hq, D, 8192, "cuda")
        out = ops.decode(q, lens, bt.cuda(), kc, vc, D ** -0.5, workspace=ws)
        got.append((out, int(ws.lean_meta[LEAN_META0 + B + 1])))
    assert got[0][1] == got[1][1] and torch.equal(got[0][0], got[1][0])
    waves = torch.cuda.get_device_properties(0).multi_processor_count * 2 // Hkv * 4
    if waves == 256:                                  # the rule's lines are shares of the waves a head has
        assert got[0][1] == max(least, -(-max(nb) // 15))
    ref = ops.decode(q.cpu(), lens.cpu(), bt, kc.cpu(), vc.cpu(), D ** -0.5)
    assert float((got[1][0].cpu().float() - ref.float()).norm() / ref.float().norm()) < 8e-3
