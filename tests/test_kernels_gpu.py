"""Numerics of every HIP kernel vs a plain PyTorch fp32 reference of the same op (run on MI355X).

Each test builds bf16 inputs on the GPU, runs the native kernel (ops dispatch to HIP for CUDA
tensors) and compares against the reference implementation evaluated on CPU copies.
"""
import math

import pytest
import torch

from financial_chatbot_llm_amd import ops
from financial_chatbot_llm_amd.ops import _native
from financial_chatbot_llm_amd.ops.attention import KV_BS, gather_kv_ref

pytestmark = pytest.mark.gpu
DEV = "cuda"


def rnd(*shape, scale=1.0, dtype=torch.bfloat16, gen=None):
    return (torch.randn(*shape, generator=gen) * scale).to(dtype)


def close(a, b, atol, rtol=0.02):
    a, b = a.float().cpu(), b.float().cpu()
    err = (a - b).abs()
    tol = atol + rtol * b.abs()
    assert bool((err <= tol).all()), f"max err {err.max().item():.4g} (atol {atol})"


def test_native_library_loaded():
    assert _native.available()
    import os
    maps = open(f"/proc/{os.getpid()}/maps").read()
    assert "libpenny_kernels.so" in maps


@pytest.mark.parametrize("T,H", [(1, 4096), (37, 4096), (64, 8192), (5, 768), (130, 2048), (5000, 4096), (3, 512)])
def test_rmsnorm(T, H):
    torch.manual_seed(0)
    x, res, w = rnd(T, H), rnd(T, H), rnd(H, scale=0.1) + 1
    y = ops.rms_norm(x.to(DEV), w.to(DEV), 1e-5)
    close(y, ops.rms_norm(x, w, 1e-5), atol=2e-2)
    r_dev = res.to(DEV)
    y2 = ops.rms_norm(x.to(DEV), w.to(DEV), 1e-5, residual=r_dev)
    r_ref = res.clone()
    y2_ref = ops.rms_norm(x, w, 1e-5, residual=r_ref)
    close(r_dev, r_ref, atol=1e-2)
    close(y2, y2_ref, atol=2e-2)


@pytest.mark.parametrize("T,H", [(3, 768), (50, 1024), (4099, 768), (7, 200), (9, 4096)])
@pytest.mark.parametrize("with_res", [True, False])
def test_layernorm(T, H, with_res):
    """wave-per-row kernel (H % 256 == 0) and the block kernel (other H) vs the f32 reference"""
    torch.manual_seed(1)
    x, r, g, b = rnd(T, H), rnd(T, H), rnd(H) * 0.1 + 1, rnd(H) * 0.1
    r = r if with_res else None
    close(ops.layer_norm(x.to(DEV), g.to(DEV), b.to(DEV), 1e-12, residual=r.to(DEV) if with_res else None),
          ops.layer_norm(x, g, b, 1e-12, residual=r), atol=3e-2)


def test_silu_mul_gelu_embedding():
    torch.manual_seed(2)
    gu = rnd(19, 2 * 1024)
    close(ops.silu_mul(gu.to(DEV)), ops.silu_mul(gu), atol=2e-2)
    x = rnd(7, 3072)
    close(ops.gelu_(x.to(DEV).clone()), ops.gelu_(x.clone()), atol=2e-2)
    table = rnd(1000, 256)
    ids = torch.randint(0, 1000, (33,))
    close(ops.embedding(ids.to(DEV), table.to(DEV)), ops.embedding(ids, table), atol=0)
    close(ops.embedding(ids.to(DEV), table[500:].to(DEV).contiguous(), 500, 1000),
          ops.embedding(ids, table[500:].contiguous(), 500, 1000), atol=0)


def _paged_setup(seq_lens, Hkv, D, num_blocks=None, gen=None):
    nb_each = [(L + KV_BS - 1) // KV_BS for L in seq_lens]
    num_blocks = num_blocks or sum(nb_each) + 3
    perm = torch.randperm(num_blocks, generator=gen)
    tables = torch.zeros((len(seq_lens), max(nb_each)), dtype=torch.int32)
    k = 0
    for i, n in enumerate(nb_each):
        tables[i, :n] = perm[k:k + n].to(torch.int32)
        k += n
    kc = rnd(num_blocks, Hkv, KV_BS * D, gen=gen)
    vc = rnd(num_blocks, Hkv, KV_BS * D, gen=gen)
    return tables, kc, vc


@pytest.mark.parametrize("Hq,Hkv,D", [(32, 8, 128), (8, 1, 128), (12, 12, 64)])
def test_rope_kv_write(Hq, Hkv, D):
    g = torch.Generator().manual_seed(3)
    T = 70
    qkv = rnd(T, (Hq + 2 * Hkv) * D, gen=g)
    pos = torch.randint(0, 4000, (T,), generator=g, dtype=torch.int32)
    cs = ops.rope_cos_sin(D, 4096, 500000.0)
    nblk = 4
    slots = torch.randperm(nblk * KV_BS, generator=g)[:T].to(torch.int32)
    slots[5] = -1
    kc = torch.zeros(nblk, Hkv, KV_BS * D, dtype=torch.bfloat16)
    vc = torch.zeros(nblk, Hkv, KV_BS * D, dtype=torch.bfloat16)
    kcd, vcd = kc.to(DEV), vc.to(DEV)
    apply = D == 128
    q = ops.rope_kv_write(qkv.to(DEV), pos.to(DEV), cs.to(DEV), slots.to(DEV), kcd, vcd, Hq, Hkv, D, apply)
    qr = ops.rope_kv_write(qkv, pos, cs, slots, kc, vc, Hq, Hkv, D, apply)
    close(q, qr, atol=2e-2)
    close(kcd, kc, atol=2e-2)
    close(vcd, vc, atol=0)


@pytest.mark.parametrize("Hq,Hkv,D,causal,lens,qscale", [
    (32, 8, 128, True, [(130, 130), (1, 77), (64, 200), (300, 300)], 1.0),   # (q_len, ctx_len): prefix hits
    (8, 1, 128, True, [(100, 100), (17, 600)], 1.0),                          # GQA 8 (70B TP=8 shard)
    (12, 12, 64, False, [(9, 9), (64, 64), (200, 200)], 1.0),                 # BERT: bidirectional, D=64
    # peaky scores (std ~12 in log2 units): exercises the deferred-max rescale path
    (32, 8, 128, True, [(700, 900), (33, 33)], 12.0),
    (32, 8, 128, False, [(257, 257)], 12.0),
])
def test_prefill_attention(Hq, Hkv, D, causal, lens, qscale):
    g = torch.Generator().manual_seed(4)
    qlens = [a for a, _ in lens]
    ctx = [b for _, b in lens]
    tables, kc, vc = _paged_setup(ctx, Hkv, D, gen=g)
    cu = torch.tensor([0] + list(torch.tensor(qlens).cumsum(0)), dtype=torch.int32)
    q = rnd(int(cu[-1]), Hq, D, scale=qscale, gen=g)
    ctx_t = torch.tensor(ctx, dtype=torch.int32)
    scale = 1 / math.sqrt(D)
    out = ops.prefill(q.to(DEV), cu.to(DEV), ctx_t.to(DEV), tables.to(DEV), kc.to(DEV), vc.to(DEV), scale, causal,
                      max_q_len=max(qlens))
    ref = ops.prefill(q, cu, ctx_t, tables, kc, vc, scale, causal)
    close(out, ref, atol=2e-2)


@pytest.mark.parametrize("variant", [4, 5, 6, 7])
@pytest.mark.parametrize("Hq,Hkv,D,causal,lens,qscale", [
    # respond chunk behind a cached prefix + decide-like and spec-like chunks (dead waves: 17 x 4 rows)
    (32, 8, 128, True, [(300, 1100), (17, 900), (70, 70), (130, 700)], 1.0),
    (32, 8, 128, True, [(257, 257), (64, 3000)], 12.0),      # rescale path, one block per op
    (8, 1, 128, True, [(40, 40), (33, 500)], 1.0),            # G = 8
    (12, 12, 64, False, [(200, 200), (33, 33)], 1.0),         # bidirectional, D = 64
])
def test_prefill_attention_big_tile_variants(variant, Hq, Hkv, D, causal, lens, qscale):
    """prefill2 with pinned fragment prefetch (4), its VALU-lean softmax (5: ones-MFMA
    row sums, lean max / grow logic) and 5 with prescaled Q and -m accumulator starts (6) vs the fp32
    reference, with the LPT work list and without (also the lse output)."""
    g = torch.Generator().manual_seed(40 + variant)
    qlens = [a for a, _ in lens]
    ctx = [b for _, b in lens]
    tables, kc, vc = _paged_setup(ctx, Hkv, D, gen=g)
    cu = torch.tensor([0] + list(torch.tensor(qlens).cumsum(0)), dtype=torch.int32)
    q = rnd(int(cu[-1]), Hq, D, scale=qscale, gen=g)
    ctx_t = torch.tensor(ctx, dtype=torch.int32)
    scale = 1 / math.sqrt(D)
    ref = ops.prefill(q, cu, ctx_t, tables, kc, vc, scale, causal)
    lse_ref = torch.empty(q.shape[0], Hq)
    ops.prefill(q, cu, ctx_t, tables, kc, vc, scale, causal, lse=lse_ref)
    wl = ops.attention.prefill_work_list(cu.numpy(), ctx_t.numpy(), Hq // Hkv, causal)
    old = ops.attention.prefill_variant(variant)
    # variant 6 rounds q*scale*log2(e) to bf16 once (opt-in): on the peaky rows (qscale 12, scores of
    # std ~17 log2 units) that perturbation shows as up to ~0.08 in the output; typical rows hold 0.02
    atol = 1e-1 if (variant == 6 and qscale > 1) else 2e-2
    try:
        for work in (None, torch.from_numpy(wl).to(DEV) if wl is not None else None):
            lse = torch.empty(q.shape[0], Hq, device=DEV)
            out = ops.prefill(q.to(DEV), cu.to(DEV), ctx_t.to(DEV), tables.to(DEV), kc.to(DEV), vc.to(DEV), scale,
                              causal, max_q_len=max(qlens), lse=lse, work=work)
            close(out, ref, atol=atol)
            close(lse, lse_ref, atol=atol, rtol=1e-3)
    finally:
        ops.attention.prefill_variant(old)


@pytest.mark.parametrize("variant", [4, 5, 6, 7])
@pytest.mark.parametrize("min_chunk", [1, 3, 8])
@pytest.mark.parametrize("Hq,Hkv,D,causal,lens", [
    (32, 8, 128, True, [(300, 1100), (9, 900), (70, 70), (130, 2000)]),   # respond / spec / first turn / decide
    (32, 8, 128, True, [(9, 3000), (2, 2100), (5, 700), (1, 1300)]),      # tiny chunks only (spec / known runs)
    (8, 1, 128, True, [(40, 1500), (33, 500)]),
    (12, 12, 64, False, [(200, 700), (33, 33)]),
])
def test_prefill_attention_lean_split_kv(variant, min_chunk, Hq, Hkv, D, causal, lens, monkeypatch):
    """Lean prefill: the KV walks of long tiles cut into chunks on different workgroups, partial
    (O, m, l) merged in chunk order -- vs the fp32 reference (output and lse), on every prefill2
    variant (the planner's cost gate off: these small steps exercise the split path by force; a
    tiny-chunks-only step reaches the split path only through the gate, which takes it here)."""
    if max(a for a, _ in lens) * (Hq // Hkv) > 128:
        monkeypatch.setattr(ops.attention, "LEAN_COST_GATE", False)
    g = torch.Generator().manual_seed(50 + min_chunk)
    qlens = [a for a, _ in lens]
    ctx = [b for _, b in lens]
    tables, kc, vc = _paged_setup(ctx, Hkv, D, gen=g)
    cu = torch.tensor([0] + list(torch.tensor(qlens).cumsum(0)), dtype=torch.int32)
    q = rnd(int(cu[-1]), Hq, D, gen=g)
    ctx_t = torch.tensor(ctx, dtype=torch.int32)
    scale = 1 / math.sqrt(D)
    ref = ops.prefill(q, cu, ctx_t, tables, kc, vc, scale, causal)
    lse_ref = torch.empty(q.shape[0], Hq)
    ops.prefill(q, cu, ctx_t, tables, kc, vc, scale, causal, lse=lse_ref)
    wl = ops.attention.prefill_lean_list(cu.numpy(), ctx_t.numpy(), Hq // Hkv, Hkv, causal, cus=100000,
                                         min_chunk=min_chunk)
    assert wl is not None and int(wl[0, 2]) > 0                 # some tiles were split
    lse = torch.empty(q.shape[0], Hq, device=DEV)
    old = ops.attention.prefill_variant(variant)
    try:
        out = ops.prefill(q.to(DEV), cu.to(DEV), ctx_t.to(DEV), tables.to(DEV), kc.to(DEV), vc.to(DEV), scale, causal,
                          max_q_len=max(qlens), lse=lse, work=torch.from_numpy(wl).to(DEV),
                          lean=(int(wl[0, 1]), int(wl[0, 2]), int(wl[0, 3])))
    finally:
        ops.attention.prefill_variant(old)
    close(out, ref, atol=2e-2)
    close(lse, lse_ref, atol=2e-2, rtol=1e-3)


@pytest.mark.parametrize("variant", [4, 5, 6, 7])
@pytest.mark.parametrize("spike_block", [0, 3, 9])
def test_prefill_attention_late_max_spike_forces_rescale(variant, spike_block):
    """Rule 26: a rare rescale branch needs an input that FORCES it.  One query token's row is made to
    match one key of block `spike_block` (score ~ 20 above every other in log2 units) so the running
    max jumps past the defer threshold exactly there, after earlier blocks already summed into O and
    l; the output must still equal the fp32 reference (every row, incl. the spiked one)."""
    from financial_chatbot_llm_amd.ops.attention import gather_kv_ref
    g = torch.Generator().manual_seed(70 + spike_block)
    Hq, Hkv, D = 32, 8, 128
    lens = [(96, 12 * 64), (40, 40)]
    qlens = [a for a, _ in lens]
    ctx = [b for _, b in lens]
    tables, kc, vc = _paged_setup(ctx, Hkv, D, gen=g)
    cu = torch.tensor([0] + list(torch.tensor(qlens).cumsum(0)), dtype=torch.int32)
    q = rnd(int(cu[-1]), Hq, D, scale=0.3, gen=g)
    # query token 90 of sequence 0 (position 762), head 5 (kv head 1) := 3.5 x key 64*spike_block + 7
    kfull, _ = gather_kv_ref(kc, vc, tables[0], ctx[0])
    key = 64 * spike_block + 7
    q[90, 5] = (kfull[key, 1].float() * 3.5).to(torch.bfloat16)
    ctx_t = torch.tensor(ctx, dtype=torch.int32)
    scale = 1 / math.sqrt(D)
    ref = ops.prefill(q, cu, ctx_t, tables, kc, vc, scale, True)
    old = ops.attention.prefill_variant(variant)
    try:
        wl = ops.attention.prefill_work_list(cu.numpy(), ctx_t.numpy(), Hq // Hkv, True)
        out = ops.prefill(q.to(DEV), cu.to(DEV), ctx_t.to(DEV), tables.to(DEV), kc.to(DEV), vc.to(DEV), scale, True,
                          max_q_len=max(qlens), work=torch.from_numpy(wl).to(DEV) if wl is not None else None)
    finally:
        ops.attention.prefill_variant(old)
    close(out, ref, atol=2e-2)
    close(out[90, 5], ref[90, 5], atol=1e-2)


@pytest.mark.parametrize("variant", [5, 7])
@pytest.mark.parametrize("spike_block", [0, 1, 4, 9])
def test_prefill_prescaled_late_spike(variant, spike_block, monkeypatch):
    """The production prescaled-Q path (7: the 32x32x16 kernel whose S^T chains start at -m; 5: the
    16x16 fold) on a FORCED late rescale: one query row matched to a key of block `spike_block`, plain
    and lean (split-KV) work lists."""
    from financial_chatbot_llm_amd.ops.attention import gather_kv_ref
    monkeypatch.setattr(ops.attention, "LEAN_COST_GATE", False)
    g = torch.Generator().manual_seed(90 + spike_block)
    Hq, Hkv, D = 32, 8, 128
    lens = [(96, 12 * 64), (40, 40), (33, 700)]
    qlens = [a for a, _ in lens]
    ctx = [b for _, b in lens]
    tables, kc, vc = _paged_setup(ctx, Hkv, D, gen=g)
    cu = torch.tensor([0] + list(torch.tensor(qlens).cumsum(0)), dtype=torch.int32)
    qf = torch.randn(int(cu[-1]), Hq, D, generator=g) * 0.3
    kfull, _ = gather_kv_ref(kc, vc, tables[0], ctx[0])
    qf[90, 5] = kfull[64 * spike_block + 7, 1].float() * 3.5
    ctx_t = torch.tensor(ctx, dtype=torch.int32)
    scale = 1 / math.sqrt(D)
    ref = ops.prefill(qf, cu, ctx_t, tables, kc, vc, scale, True)
    qp = (qf * (scale * 1.4426950408889634)).to(torch.bfloat16)
    args = (cu.to(DEV), ctx_t.to(DEV), tables.to(DEV), kc.to(DEV), vc.to(DEV))
    old = ops.attention.prefill_variant(variant)
    try:
        out = ops.prefill(qp.to(DEV), *args, 1 / 1.4426950408889634, True, max_q_len=max(qlens), q_prescaled=True)
        wl = ops.attention.prefill_lean_list(cu.numpy(), ctx_t.numpy(), Hq // Hkv, Hkv, True, cus=100000,
                                             min_chunk=1)
        outl = ops.prefill(qp.to(DEV), *args, 1 / 1.4426950408889634, True, max_q_len=max(qlens),
                           work=torch.from_numpy(wl).to(DEV), lean=(int(wl[0, 1]), int(wl[0, 2]), int(wl[0, 3])),
                           q_prescaled=True)
    finally:
        ops.attention.prefill_variant(old)
    for o in (out, outl):
        close(o, ref, atol=3e-2)
        close(o[90, 5], ref[90, 5], atol=2e-2)


@pytest.mark.parametrize("Hq,Hkv,ctxs", [(32, 8, [1, 63, 64, 65, 700, 2100]), (8, 1, [5, 1500]), (64, 8, [333]),
                                         # B >= 96 / >= 192: longer partitions (pb 16 / 32)
                                         (32, 8, [(37 * i) % 3000 + 1 for i in range(100)]),
                                         (8, 2, [(53 * i) % 4000 + 1 for i in range(200)]),
                                         # lean split: one long row among short ones, many rows
                                         (32, 8, [8000] + [70] * 40 + [3000, 1]),
                                         (32, 8, [(97 * i) % 500 + 1 for i in range(700)])])
@pytest.mark.parametrize("lean", [True, False])
def test_decode_attention(Hq, Hkv, ctxs, lean, monkeypatch):
    monkeypatch.setattr(ops.attention, "DECODE_LEAN", lean)
    g = torch.Generator().manual_seed(5)
    D = 128
    tables, kc, vc = _paged_setup(ctxs, Hkv, D, gen=g)
    q = rnd(len(ctxs), Hq, D, gen=g)
    ctx_t = torch.tensor(ctxs, dtype=torch.int32)
    scale = 1 / math.sqrt(D)
    ws = ops.DecodeWorkspace.create(len(ctxs), Hq, D, max(ctxs), DEV)
    out = ops.decode(q.to(DEV), ctx_t.to(DEV), tables.to(DEV), kc.to(DEV), vc.to(DEV), scale, workspace=ws)
    ref = ops.decode(q, ctx_t, tables, kc, vc, scale)
    close(out, ref, atol=2e-2)


def test_prefill_work_list_matches_grid_order():
    """LPT work list (one workgroup per real (sequence, tile), longest KV walk first) gives the
    same attention as the (max tiles x sequences) grid, bitwise."""
    g = torch.Generator().manual_seed(9)
    Hq, Hkv, D = 32, 8, 128
    lens = [(1600, 3400)] + [(220, 4600)] * 3 + [(9, 5000), (300, 300)]
    ctx = [c for _, c in lens]
    tables, kc, vc = _paged_setup(ctx, Hkv, D, gen=g)
    cu = torch.tensor([0] + list(torch.tensor([a for a, _ in lens]).cumsum(0)), dtype=torch.int32)
    q = rnd(int(cu[-1]), Hq, D, gen=g)
    ctx_t = torch.tensor(ctx, dtype=torch.int32)
    work = ops.attention.prefill_work_list(cu.numpy(), ctx_t.numpy(), Hq // Hkv)
    assert work is not None and len(work) == 25 + 3 * 4 + 1 + 5
    args = (q.to(DEV), cu.to(DEV), ctx_t.to(DEV), tables.to(DEV), kc.to(DEV), vc.to(DEV), 0.088, True, 1600)
    a = ops.prefill(*args)
    b = ops.prefill(*args, work=torch.from_numpy(work).to(DEV))
    assert torch.equal(a, b)
    close(b, ops.prefill(q, cu, ctx_t, tables, kc, vc, 0.088, True), atol=2e-2)


def test_decode_matches_prefill_last_row():
    g = torch.Generator().manual_seed(6)
    Hq, Hkv, D, L = 32, 8, 128, 517
    tables, kc, vc = _paged_setup([L], Hkv, D, gen=g)
    q = rnd(L, Hq, D, gen=g)
    cu = torch.tensor([0, L], dtype=torch.int32)
    ctx = torch.tensor([L], dtype=torch.int32)
    a = ops.prefill(q.to(DEV), cu.to(DEV), ctx.to(DEV), tables.to(DEV), kc.to(DEV), vc.to(DEV), 0.088, True, L)
    b = ops.decode(q[-1:].to(DEV), ctx.to(DEV), tables.to(DEV), kc.to(DEV), vc.to(DEV), 0.088)
    close(a[-1:], b, atol=2e-2)


def test_sampler_greedy_and_distribution():
    torch.manual_seed(7)
    V = 128256
    logits = rnd(6, V, scale=3.0)
    temps = torch.tensor([0.0, 0.0, 0.5, 1.0, 0.0, 2.0])
    seeds = torch.arange(6, dtype=torch.int64) * 7919
    ids = ops.sample(logits.to(DEV), temps.to(DEV), seeds.to(DEV)).cpu()
    for b in (0, 1, 4):
        assert int(ids[b]) == int(torch.argmax(logits[b].float()))
    # distribution: many seeds over a small vocab vs softmax(l / T)
    Vs = 64
    lg = torch.linspace(-2, 2, Vs).repeat(4096, 1).to(torch.float32)
    t = torch.full((4096,), 0.5)
    sd = torch.arange(4096, dtype=torch.int64) * 104729 + 13
    draws = ops.sample(lg.to(DEV).contiguous(), t.to(DEV), sd.to(DEV)).cpu().long()
    emp = torch.bincount(draws, minlength=Vs).float() / 4096
    p = torch.softmax(lg[0] / 0.5, -1)
    assert (emp - p).abs().max() < 0.03
    # bf16 logits, determinism for a fixed seed
    again = ops.sample(logits.to(DEV), temps.to(DEV), seeds.to(DEV)).cpu()
    assert torch.equal(ids, again)


def test_filtered_topk():
    g = torch.Generator().manual_seed(8)
    N, D = 200_000, 768
    corpus = torch.nn.functional.normalize(torch.randn(N, D, generator=g), dim=-1).to(torch.bfloat16)
    users = torch.randint(0, 500, (N,), generator=g, dtype=torch.int32)
    users[:9000] = 7  # one heavy user -> exercises the > SORT_CAP path
    dates = torch.randint(0, 1_000_000, (N,), generator=g, dtype=torch.int64)
    q = torch.nn.functional.normalize(torch.randn(5, D, generator=g), dim=-1).to(torch.bfloat16)
    qu = torch.tensor([1, 2, 7, 499, 1234], dtype=torch.int32)
    qf = torch.tensor([0, 500_000, 0, -(1 << 62), 0], dtype=torch.int64)
    ks = torch.tensor([10, 10000, 50, 3, 5], dtype=torch.int32)
    kmax = 10000
    ids, sc, cnt = ops.filtered_topk(corpus.to(DEV), users.to(DEV), dates.to(DEV), q.to(DEV), qu.to(DEV),
                                     qf.to(DEV), ks.to(DEV), kmax)
    rids, rsc, rcnt = ops.filtered_topk(corpus, users, dates, q, qu, qf, ks, kmax)
    assert cnt.cpu().tolist() == rcnt.tolist()
    for i in range(5):
        c = int(rcnt[i])
        close(sc[i, :c], rsc[i, :c], atol=2e-3, rtol=0)
        # ids may differ only where scores tie within rounding
        same = (ids[i, :c].cpu() == rids[i, :c]).float().mean().item() if c else 1.0
        assert same > 0.97


@pytest.mark.parametrize("M", [1, 7, 16, 33, 64])
@pytest.mark.parametrize("cfg", [(2, 4), (2, 8), (4, 4), (1, 8)])
def test_skinny_gemm(M, cfg):
    from financial_chatbot_llm_amd.ops import gemm
    g = torch.Generator().manual_seed(9)
    N_, K = 512, 2048
    x = rnd(M, K, gen=g)
    w = rnd(N_, K, scale=0.05, gen=g)
    gemm.TUNING[(N_, K)] = cfg
    try:
        y = gemm.linear(x.to(DEV), w.to(DEV), wt=gemm.tile_weight(w.to(DEV)))
        ref = (x.float() @ w.float().t())
        close(y, ref, atol=2e-2)
        if cfg[0] % 2 == 0:
            gate, up = w[:256], w[256:]
            wi = gemm.interleave16(gate, up)
            wid = wi.to(DEV).contiguous()
            y2 = gemm.linear(x.to(DEV), wid, epilogue="silu", wt=gemm.tile_weight(wid))
            ref2 = ops.silu_mul(torch.cat([(x.float() @ gate.float().t()), (x.float() @ up.float().t())], -1).to(torch.bfloat16))
            close(y2, ref2, atol=3e-2)
    finally:
        gemm.TUNING.pop((N_, K), None)


def _paired(fn):
    """fn() with the decode GEMM streams issuing their BK=64 stages in pairs (gemm.PAIR_MODE)."""
    from financial_chatbot_llm_amd.ops import gemm
    gemm.PAIR_MODE = "1"
    try:
        return fn()
    finally:
        gemm.PAIR_MODE = "table"


@pytest.mark.parametrize("M", [5, 33, 64, 90, 128, 200, 256])
@pytest.mark.parametrize("S,nf", [(1, 4), (2, 8), (4, 4), (8, 8), (2, 2), (4, 6)])
def test_splitk_gemm(M, S, nf):
    """Mid-batch split-K GEMM (f32 slabs) + slab reduce (+ residual) vs the fp32 reference."""
    from financial_chatbot_llm_amd.ops import gemm
    g = torch.Generator().manual_seed(11)
    N_, K = 384, 2048
    x = rnd(M, K, gen=g)
    w = rnd(N_, K, scale=0.05, gen=g)
    res = rnd(M, N_, gen=g)
    wt = gemm.tile_weight(w.to(DEV))
    P = gemm.splitk_partials(x.to(DEV), wt, N_, S, nf)
    ref_p = (x.float().view(M, S, K // S).transpose(0, 1) @ w.float().view(N_, S, K // S).permute(1, 2, 0))
    close(P, ref_p, atol=1e-3)
    # the row-major weight (no tiled copy) runs the identical MFMA sequence: bit-equal slabs
    assert torch.equal(gemm.splitk_partials(x.to(DEV), w.to(DEV), N_, S, nf, rowmajor=True), P)
    # ... and so does the paired-stage row-major stream (same k order)
    assert torch.equal(_paired(lambda: gemm.splitk_partials(x.to(DEV), w.to(DEV), N_, S, nf, rowmajor=True)), P)
    assert torch.equal(_paired(lambda: gemm.splitk_partials(x.to(DEV), wt, N_, S, nf)), P)
    close(gemm.splitk_reduce(P), x.float() @ w.float().t(), atol=2e-2)
    close(gemm.splitk_reduce(P, residual=res.to(DEV)), x.float() @ w.float().t() + res.float(), atol=3e-2)
    # strided X (a view into a wider activation buffer) is a supported input
    xw = torch.zeros(M, K + 64, dtype=torch.bfloat16)
    xw[:, 32:32 + K] = x
    P2 = gemm.splitk_partials(xw.to(DEV)[:, 32:32 + K], wt, N_, S, nf)
    close(P2, ref_p, atol=1e-3)


@pytest.mark.parametrize("M", [257, 600, 1100])
def test_splitk_kernels_token_chunks(M):
    """M > 256 on the decode kernels: 256-row token chunks side by side (grid y) -- slabs, bf16 output
    and the fused gate|up, row-major and fragment-tiled W, single and paired stages, vs fp32."""
    from financial_chatbot_llm_amd.ops import gemm
    g = torch.Generator().manual_seed(21)
    N_, K = 512, 1024
    x = rnd(M, K, gen=g).to(DEV)
    w = rnd(N_, K, scale=0.05, gen=g).to(DEV)
    wt = gemm.tile_weight(w)
    ref = x.float() @ w.float().t()
    for S, nf in ((1, 4), (2, 8), (4, 2)):
        P = gemm.splitk_partials(x, wt, N_, S, nf)
        close(P.sum(0), ref, atol=2e-3)
        assert torch.equal(gemm.splitk_partials(x, w, N_, S, nf, rowmajor=True), P)
        assert torch.equal(_paired(lambda: gemm.splitk_partials(x, wt, N_, S, nf)), P)
    for nf in (2, 4, 8):
        y = gemm.splitk_bf16(x, w, N_, nf)
        close(y, ref, atol=2e-2)
        assert torch.equal(gemm.splitk_bf16(x, wt, N_, nf, rowmajor=False), y)
    gate, up = rnd(N_ // 2, K, scale=0.05, gen=g).to(DEV), rnd(N_ // 2, K, scale=0.05, gen=g).to(DEV)
    wi = gemm.interleave16(gate, up).contiguous()
    ys = torch.nn.functional.silu(x.float() @ gate.float().t()) * (x.float() @ up.float().t())
    for nf in (2, 4, 8):
        yg = gemm.gateup_silu(x, gemm.tile_weight(wi), N_, nf)
        close(yg, ys, atol=3e-2)
        assert torch.equal(gemm.gateup_silu(x, wi, N_, nf, rowmajor=True), yg)


def test_linear_tp8_o_shard_small_prefill_on_chunked_kernel(monkeypatch):
    """The 70B TP=8 O shard at a 384-row prefill step: the chunked bf16 decode kernel (policy K4,
    r5) and the r6 128 x 128 tile kernel (policy M1, what the policy takes now) both equal the fp32
    reference."""
    from financial_chatbot_llm_amd.ops import gemm
    monkeypatch.delenv("PENNY_PREFILL_GEMM", raising=False)
    assert gemm.prefill_choice(384, 8192, 1024, None) == "M1"
    g = torch.Generator().manual_seed(31)
    x = rnd(384, 1024, gen=g).to(DEV)
    w = rnd(8192, 1024, scale=0.03, gen=g).to(DEV)
    y = gemm.linear(x, w)
    close(y, x.float() @ w.float().t(), atol=2e-2)
    close(y, torch.nn.functional.linear(x, w), atol=2e-2)
    close(gemm.splitk_bf16(x, w, 8192, 4), x.float() @ w.float().t(), atol=2e-2)      # the r5 K4 form


@pytest.mark.parametrize("N_,K,S,nf", [(1280, 8192, 8, 4), (8192, 8192, 4, 8), (8192, 3584, 2, 4)])
def test_splitk_rowmajor_tp_and_70b_shapes(N_, K, S, nf):
    """The table shapes that stream the row-major weight (70B, TP=8 shards) vs the fp32 reference."""
    from financial_chatbot_llm_amd.ops import gemm
    g = torch.Generator().manual_seed(8)
    x = rnd(96, K, gen=g).to(DEV)
    w = rnd(N_, K, scale=0.02, gen=g).to(DEV)
    y = gemm.splitk_reduce(gemm.splitk_partials(x, w, N_, S, nf, rowmajor=True))
    close(y, x.float() @ w.float().t(), atol=3e-2)
    assert torch.equal(_paired(lambda: gemm.splitk_reduce(gemm.splitk_partials(x, w, N_, S, nf, rowmajor=True))), y)
    for nf2 in (2, 4, 8):          # the bf16-output (row-parallel TP shard) form
        yb = gemm.splitk_bf16(x, w, N_, nf2)
        close(yb, x.float() @ w.float().t(), atol=3e-2)
        assert torch.equal(_paired(lambda: gemm.splitk_bf16(x, w, N_, nf2)), yb)


@pytest.mark.parametrize("M,F", [(1, 384), (37, 14336), (300, 2048)])
def test_silu_quant_rows_fp8_matches_two_pass(M, F):
    """Fused SiLU*up + per-row fp8 quantisation == silu_mul then quant_rows (same arithmetic)."""
    from financial_chatbot_llm_amd.ops import moe
    g = torch.Generator().manual_seed(4)
    gu = rnd(M, 2 * F, gen=g).to(DEV)
    q1, s1 = moe.silu_quant_rows_fp8(gu)
    q2, s2 = moe.quant_rows_fp8(ops.silu_mul(gu, interleave16=True))
    assert torch.equal(s1, s2)
    assert torch.equal(q1.view(torch.uint8), q2.view(torch.uint8))


@pytest.mark.parametrize("T,k", [(1, 2), (37, 2), (300, 2), (64, 1)])
def test_moe_combine_weighted(T, k):
    """Prefill MoE combine: weighted gather over the expert-sorted rows == scaled index_add."""
    from financial_chatbot_llm_amd.ops import moe
    g = torch.Generator().manual_seed(3)
    E, H = 8, 512
    logits = torch.randn(T, E, generator=g)
    topw, topi = moe.topk_softmax(logits, k)
    order, offsets, tok_idx, tok_w = moe.route(topi.to(DEV), topw.to(DEV), E)
    ys = rnd(T * k, H, gen=g).to(DEV)
    ref = torch.zeros(T, H, dtype=torch.float32, device=DEV)
    ref.index_add_(0, tok_idx, ys.float() * tok_w[:, None])
    close(moe.combine_weighted(ys, order, tok_w, T, k), ref, atol=2e-2)


@pytest.mark.parametrize("M", [1, 17, 48, 100, 128, 256])
@pytest.mark.parametrize("nf", [4, 8])
def test_gateup_silu_gemm(M, nf):
    """Fused gate|up GEMM + SiLU*up (interleave16 weight, fragment-tiled) vs the fp32 reference
    silu(x gate^T) * (x up^T), and vs the unfused hipBLASLt + silu_mul path it replaces."""
    from financial_chatbot_llm_amd.ops import gemm
    g = torch.Generator().manual_seed(5)
    Fr, K = 512, 1024
    x = rnd(M, K, gen=g)
    gate, up = rnd(Fr, K, scale=0.05, gen=g), rnd(Fr, K, scale=0.05, gen=g)
    wi = gemm.interleave16(gate, up).to(DEV).contiguous()
    y = gemm.gateup_silu(x.to(DEV), gemm.tile_weight(wi), 2 * Fr, nf)
    assert torch.equal(gemm.gateup_silu(x.to(DEV), wi, 2 * Fr, nf, rowmajor=True), y)
    assert torch.equal(_paired(lambda: gemm.gateup_silu(x.to(DEV), wi, 2 * Fr, nf, rowmajor=True)), y)
    assert torch.equal(_paired(lambda: gemm.gateup_silu(x.to(DEV), gemm.tile_weight(wi), 2 * Fr, nf)), y)
    gf, uf = x.float() @ gate.float().t(), x.float() @ up.float().t()
    close(y, torch.nn.functional.silu(gf) * uf, atol=3e-2)
    unfused = ops.silu_mul(torch.nn.functional.linear(x.to(DEV), wi), interleave16=True)
    close(y, unfused, atol=2e-2)
    # strided X is a supported input; output rows land at the given stride
    xw = torch.zeros(M, K + 64, dtype=torch.bfloat16)
    xw[:, 32:32 + K] = x
    out = torch.zeros(M, Fr + 8, dtype=torch.bfloat16, device=DEV)
    gemm.gateup_silu(xw.to(DEV)[:, 32:32 + K], gemm.tile_weight(wi), 2 * Fr, nf, out=out[:, :Fr])
    close(out[:, :Fr], y, atol=0, rtol=0)
    assert (out[:, Fr:] == 0).all()


@pytest.mark.parametrize("S,T", [(1, 3), (4, 128), (8, 200)])
def test_slab_consumers_match_reduce_then_op(S, T):
    """RMSNorm (+residual) and RoPE/KV-write fed the split-K slabs directly equal the same kernels
    fed the reduced bf16 activation -- the fused reduction rounds exactly where the GEMM would."""
    from financial_chatbot_llm_amd.ops.gemm import Slabs, splitk_reduce
    g = torch.Generator().manual_seed(12)
    H = 4096
    P = (torch.randn(S, T, H, generator=g) * 0.3).to(DEV)
    w = (rnd(H, scale=0.1, gen=g) + 1).to(DEV)
    res = rnd(T, H, gen=g).to(DEV)
    r1, r2 = res.clone(), res.clone()
    y1 = ops.rms_norm(Slabs(P), w, 1e-5, residual=r1)
    y2 = ops.rms_norm(splitk_reduce(P), w, 1e-5, residual=r2)
    close(y1, y2, atol=1e-6, rtol=0)
    close(r1, r2, atol=0, rtol=0)
    close(ops.rms_norm(Slabs(P), w, 1e-5), ops.rms_norm(splitk_reduce(P), w, 1e-5), atol=1e-6, rtol=0)
    Hq, Hkv, D = 32, 8, 128
    W = (Hq + 2 * Hkv) * D
    Pq = (torch.randn(S, T, W, generator=g) * 0.3).to(DEV)
    pos = torch.randint(0, 4000, (T,), generator=g, dtype=torch.int32).to(DEV)
    cs = ops.rope_cos_sin(D, 4096, 500000.0).to(DEV)
    nblk = (T + KV_BS - 1) // KV_BS + 1
    slots = torch.randperm(nblk * KV_BS, generator=g)[:T].to(torch.int32).to(DEV)
    kc1, vc1 = (torch.zeros(nblk, Hkv, KV_BS * D, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    kc2, vc2 = kc1.clone(), vc1.clone()
    q1 = ops.rope_kv_write(Slabs(Pq), pos, cs, slots, kc1, vc1, Hq, Hkv, D)
    q2 = ops.rope_kv_write(splitk_reduce(Pq), pos, cs, slots, kc2, vc2, Hq, Hkv, D)
    # q/k: the rotation's FMA contraction may differ between the two instantiations -> 1 bf16 ulp
    close(q1, q2, atol=1e-6, rtol=2 ** -7)
    close(kc1, kc2, atol=1e-6, rtol=2 ** -7)
    close(vc1, vc2, atol=0, rtol=0)


def test_silu_mul_interleaved():
    from financial_chatbot_llm_amd.ops import gemm
    g = torch.Generator().manual_seed(10)
    gate, up = rnd(13, 256, gen=g), rnd(13, 256, gen=g)
    il = gemm.interleave16(gate.t().contiguous(), up.t().contiguous()).t().contiguous()
    close(ops.silu_mul(il.to(DEV), interleave16=True), ops.silu_mul(torch.cat([gate, up], -1)), atol=2e-2)


@pytest.mark.parametrize("T", [1, 13, 64, 200])
def test_moe_fp8_pipeline(T):
    from financial_chatbot_llm_amd.ops import gemm, moe
    g = torch.Generator().manual_seed(11)
    E, H, F_, K = 8, 512, 384, 2
    h = rnd(T, H, gen=g)
    router = rnd(E, H, scale=0.2, gen=g)
    w13 = rnd(E, 2 * F_, H, scale=0.05, gen=g)
    w2 = rnd(E, H, F_, scale=0.05, gen=g)
    w13i = torch.stack([gemm.interleave16(w13[e, :F_], w13[e, F_:]) for e in range(E)])
    q13, s13 = moe.quantize_fp8_rowwise(w13i)
    q2, s2 = moe.quantize_fp8_rowwise(w2)
    ref = moe.moe_fp8_reference(h.float(), router.float(), q13, s13, q2, s2, K)
    ws = moe.MoEWorkspace(256, K, E, H, F_, DEV)
    logits = (h.to(DEV) @ router.to(DEV).t()).contiguous()
    out = moe.moe_decode_fp8(h.to(DEV), logits, moe.tile_fp8_weight(q13.to(DEV)), s13.to(DEV),
                             moe.tile_fp8_weight(q2.to(DEV)), s2.to(DEV), K, ws)
    # same arithmetic (fp8 activations, per-row scales) in fp32: only accumulation order/bf16 rounding differ
    ref_q = moe.moe_fp8_reference(h.float(), router.float(), q13, s13, q2, s2, K, quant_act=True)
    err_q = (out.float().cpu() - ref_q.float()).abs()
    assert err_q.mean() < 0.01 * ref_q.float().abs().mean() + 1e-4, (err_q.mean(), ref_q.abs().mean())
    # vs high-precision activations: two e4m3 roundings of the GEMM inputs cost ~5% relative
    err = (out.float().cpu() - ref.float()).abs()
    assert err.mean() < 0.08 * ref.float().abs().mean() + 1e-3, (err.mean(), ref.abs().mean())
    assert int(ws.offsets[-1]) == T * K


def _shared_prefix_tables(B, groups, W, num_blocks, gen):
    """Block tables where rows of each group share `lcp` leading physical blocks."""
    perm = torch.randperm(num_blocks, generator=gen).to(torch.int32)
    tables = torch.zeros((B, W), dtype=torch.int32)
    k, row = 0, 0
    for size, lcp in groups:
        shared = perm[k:k + lcp]
        k += lcp
        for _ in range(size):
            tables[row, :lcp] = shared
            tables[row, lcp:] = perm[k:k + W - lcp]
            k += W - lcp
            row += 1
    while row < B:
        tables[row] = perm[k:k + W]
        k += W
        row += 1
    return tables


@pytest.mark.parametrize("lean", [True, False])
@pytest.mark.parametrize("D,Hq,Hkv", [(128, 32, 8), (64, 8, 4)])
def test_shared_prefix_decode_matches_reference(D, Hq, Hkv, lean, monkeypatch):
    """Prefix-cached rows pointing at the SAME physical blocks: the lean kernel (default) and the
    partitioned fallback (PENNY_DECODE_LEAN=0) both equal the fp32 reference."""
    monkeypatch.setattr(ops.attention, "DECODE_LEAN", lean)
    g = torch.Generator().manual_seed(12)
    # group A: 40 rows x 10 shared blocks; group B: 5 rows x 3; 3 loners
    groups = [(40, 10), (5, 3)]
    B, W = 48, 24
    nb = 40 * 14 + 5 * 21 + 3 * W + 16
    tables = _shared_prefix_tables(B, groups, W, nb, g)
    ctx = torch.randint(1, 14 * KV_BS, (B,), generator=g, dtype=torch.int32)
    ctx[:40] = torch.randint(10 * KV_BS + 1, 14 * KV_BS, (40,), generator=g, dtype=torch.int32)
    ctx[40:45] = torch.randint(3 * KV_BS + 1, 20 * KV_BS, (5,), generator=g, dtype=torch.int32)
    kc, vc = rnd(nb, Hkv, KV_BS * D, gen=g), rnd(nb, Hkv, KV_BS * D, gen=g)
    q = rnd(B, Hq, D, gen=g)
    scale = 1 / math.sqrt(D)
    ws = ops.DecodeWorkspace.create(B, Hq, D, W * KV_BS, DEV)
    out = ops.decode(q.to(DEV), ctx.to(DEV), tables.to(DEV), kc.to(DEV), vc.to(DEV), scale, workspace=ws)
    ref = ops.decode(q, ctx, tables, kc, vc, scale)
    close(out, ref, atol=2e-2)
    # the engine's shared-block marks (-id - 1) + non-temporal loads for the unmarked blocks: the
    # cache policy changes, the result does not (bit-equal), on either decode kernel
    marked = torch.from_numpy(ops.attention.mark_shared_blocks(tables.numpy().copy(), ctx.numpy()))
    assert (marked[:40, :10] < 0).all() and (marked[45:] >= 0).all()
    monkeypatch.setattr(ops.attention, "LEAN_FLAGS", 1)
    out_m = ops.decode(q.to(DEV), ctx.to(DEV), marked.to(DEV), kc.to(DEV), vc.to(DEV), scale, workspace=ws)
    assert torch.equal(out_m, out)


def _kept_ref(lg, k, p, t):
    m = ops.apply_top_k_top_p(lg[None].float(), torch.tensor([k]), torch.tensor([p]), torch.tensor([t]))[0]
    return torch.isfinite(m)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_topk_topp_threshold_matches_reference(dtype):
    """HIP radix-select threshold vs the fp32 sort-based reference: same kept sets (up to tokens
    tied with the threshold logit), nucleus mass >= p, and k/p-off rows keep everything."""
    from financial_chatbot_llm_amd.ops.sampling import topk_topp_threshold
    g = torch.Generator().manual_seed(11)
    V = 128256
    cases = [(50, 1.0, 1.0), (0, 0.9, 0.7), (40, 0.5, 1.0), (1, 1.0, 0.5), (0, 1.0, 1.0), (1000, 0.95, 1.3),
             (0, 0.3, 0.5), (5, 0.99, 2.0)]
    lg = (torch.randn(len(cases), V, generator=g) * 3.0).to(dtype)
    k = torch.tensor([c[0] for c in cases], dtype=torch.int32)
    p = torch.tensor([c[1] for c in cases], dtype=torch.float32)
    t = torch.tensor([c[2] for c in cases], dtype=torch.float32)
    th = topk_topp_threshold(lg.to(DEV), t.to(DEV), k.to(DEV), p.to(DEV)).cpu()
    for i, (kk, pp, tt) in enumerate(cases):
        row = lg[i].float()
        kept = row >= th[i]
        ref = _kept_ref(lg[i], kk, pp, tt)
        if kk <= 0 and pp >= 1:
            assert th[i] == float("-inf")
            continue
        assert bool((kept | ~ref).all()), f"case {i}: kernel dropped a reference token"
        extra = kept & ~ref
        assert bool((row[extra] == th[i]).all()), f"case {i}: extra tokens not ties of the threshold"
        if kk > 0:
            assert int((row > th[i]).sum()) < kk
            if pp >= 1:
                assert int(kept.sum()) >= min(kk, V)
        if pp < 1:
            surv = row >= (torch.sort(row, descending=True).values[kk - 1] if kk > 0 else -float("inf"))
            probs = torch.softmax(torch.where(surv, row / tt, torch.tensor(-float("inf"))), -1)
            assert float(probs[kept].sum()) >= pp - 1e-3
            assert float(probs[row > th[i]].sum()) < pp + 1e-3


def test_sampler_with_top_k_top_p_stays_in_the_nucleus():
    V = 32000
    g = torch.Generator().manual_seed(5)
    base = torch.randn(V, generator=g) * 2
    n = 2048
    lg = base.repeat(n, 1).contiguous()
    t = torch.full((n,), 1.0)
    sd = torch.arange(n, dtype=torch.int64) * 7919 + 3
    k = torch.full((n,), 8, dtype=torch.int32)
    p = torch.ones(n)
    draws = ops.sample(lg.to(DEV), t.to(DEV), sd.to(DEV), top_k=k.to(DEV), top_p=p.to(DEV)).cpu().long()
    top8 = torch.topk(base, 8).indices
    assert bool(torch.isin(draws, top8).all())
    emp = torch.bincount(draws, minlength=V)[top8].float() / n
    want = torch.softmax(base[top8], -1)
    assert (emp - want).abs().max() < 0.05
    # top_k = 1 at any temperature == greedy
    one = ops.sample(lg[:4].to(DEV), torch.full((4,), 5.0, device=DEV), sd[:4].to(DEV),
                     top_k=torch.ones(4, dtype=torch.int32, device=DEV), top_p=torch.ones(4, device=DEV)).cpu()
    assert bool((one.long() == int(torch.argmax(base))).all())
    # nucleus: p=0.5 draws only from the smallest top set holding >= 50 % of the mass
    probs = torch.softmax(base, -1)
    sp, si = torch.sort(probs, descending=True)
    nuc = si[: int((torch.cumsum(sp, 0) < 0.5).sum()) + 1]
    draws = ops.sample(lg.to(DEV), t.to(DEV), sd.to(DEV), top_k=torch.zeros(n, dtype=torch.int32, device=DEV),
                       top_p=torch.full((n,), 0.5, device=DEV)).cpu().long()
    assert bool(torch.isin(draws, nuc).all())


def _moe_bank(g, E=8, H=512, F_=384):
    from financial_chatbot_llm_amd.ops import gemm, moe
    w13 = rnd(E, 2 * F_, H, scale=0.05, gen=g)
    w2 = rnd(E, H, F_, scale=0.05, gen=g)
    w13i = torch.stack([gemm.interleave16(w13[e, :F_], w13[e, F_:]) for e in range(E)])
    q13, s13 = moe.quantize_fp8_rowwise(w13i)
    q2, s2 = moe.quantize_fp8_rowwise(w2)
    return q13, s13, q2, s2


@pytest.mark.parametrize("T", [700, 2500])
def test_moe_prefill_fp8_device_pipeline(T):
    """Prefill-size MoE with device-side routing (no host sync): grouped fp8 MFMA GEMMs over the
    expert buckets == fp32 reference of the same fp8 arithmetic (odd T, > the route kernel's cap)."""
    from financial_chatbot_llm_amd.ops import moe
    g = torch.Generator().manual_seed(21)
    E, H, K = 8, 512, 2
    q13, s13, q2, s2 = _moe_bank(g, E, H)
    h = rnd(T, H, gen=g)
    router = rnd(E, H, scale=0.2, gen=g)
    logits = (h.to(DEV) @ router.to(DEV).t()).contiguous()
    out = moe.moe_prefill_fp8(h.to(DEV), logits, moe.tile_fp8_weight(q13.to(DEV)), s13.to(DEV),
                              moe.tile_fp8_weight(q2.to(DEV)), s2.to(DEV), K)
    ref = moe.moe_fp8_reference(h.float(), router.float(), q13, s13, q2, s2, K, quant_act=True)
    # same criterion as the decode pipeline test: an activation landing on the other side of an
    # e4m3 rounding boundary moves single outputs, so bound the mean error
    err = (out.float().cpu() - ref.float()).abs()
    assert err.mean() < 0.01 * ref.float().abs().mean() + 1e-4, (err.mean(), ref.abs().mean())


@pytest.mark.parametrize("T,E,K,H", [(1, 8, 2, 512), (3000, 8, 2, 4096), (517, 64, 6, 2048), (64, 16, 4, 6144)])
def test_moe_route_quant_matches_torch_chain(T, E, K, H):
    """penny_moe_route_quant (route + quantise in 2 launches) == topk_softmax + route_device +
    quant_rows: identical fp8 rows and scales, expert offsets, and the same (token, weight) pairs in
    each expert bucket; the inverse map points every (token, j) at a slot holding that token."""
    from financial_chatbot_llm_amd.ops import moe
    g = torch.Generator().manual_seed(31)
    h = rnd(T, H, gen=g).to(DEV)
    # distinct logits per row (a bf16 tie would leave the top-k choice to each implementation)
    perm = torch.stack([torch.randperm(E, generator=g) for _ in range(T)]).float()
    logits = ((perm - E / 2) * 0.1).to(torch.bfloat16).to(DEV)
    xq, xs, off, tok, tw, inv = moe.route_quant_device(h, logits, K, E)
    rq, rs = moe.quant_rows_fp8(h)
    assert torch.equal(xq.view(torch.uint8), rq.view(torch.uint8)) and torch.equal(xs, rs)
    topw, topi = moe.topk_softmax(logits, K)
    roff, rtok, rtw, rinv = moe.route_device(topi, topw, E)
    assert torch.equal(off.cpu(), roff.cpu())
    off = off.cpu().tolist()
    tok, tw, inv = tok.cpu(), tw.cpu(), inv.cpu()
    rtok, rtw = rtok.cpu(), rtw.cpu()
    for e in range(E):
        a, b = off[e], off[e + 1]
        mine = sorted(zip(tok[a:b].tolist(), tw[a:b].tolist()))
        ref = sorted(zip(rtok[a:b].tolist(), rtw[a:b].tolist()))
        assert [m[0] for m in mine] == [r[0] for r in ref], e
        assert max((abs(m[1] - r[1]) for m, r in zip(mine, ref)), default=0.0) < 1e-5, e
    assert torch.equal(tok[inv.long()], torch.arange(T).repeat_interleave(K).to(torch.int32))
    assert torch.equal(torch.sort(inv.long()).values, torch.arange(T * K))


def test_moe_grouped_fp8_with_padding_rows():
    """EP receive side: rows tagged with their local expert (-1 = capacity padding) in one grouped
    call == per-row fp32 reference; padding rows come back zero."""
    from financial_chatbot_llm_amd.ops import activation, moe
    g = torch.Generator().manual_seed(22)
    E, H = 4, 512
    q13, s13, q2, s2 = _moe_bank(g, E, H)
    M = 301
    x = rnd(M, H, gen=g)
    ids = torch.randint(-1, E, (M,), generator=g, dtype=torch.int32)
    y = moe.moe_grouped_fp8(x.to(DEV), ids.to(DEV), moe.tile_fp8_weight(q13.to(DEV)), s13.to(DEV),
                            moe.tile_fp8_weight(q2.to(DEV)), s2.to(DEV)).float().cpu()
    ref = torch.zeros(M, H)
    for i in range(M):
        e = int(ids[i])
        if e < 0:
            assert float(y[i].abs().max()) == 0.0
            continue
        xi = moe._fake_quant_rows(x[i:i + 1].float())
        a = activation.silu_mul((xi @ (q13[e].float() * s13[e][:, None]).t()).to(torch.bfloat16), interleave16=True)
        ref[i] = (moe._fake_quant_rows(a.float()) @ (q2[e].float() * s2[e][:, None]).t())[0]
    valid = ids >= 0
    err = (y[valid] - ref[valid]).abs()
    # e4m3 rounding-boundary flips move single rows by a few %; the aggregate matches tightly
    assert err.mean() < 0.01 * ref[valid].abs().mean() + 1e-4, (err.mean(), ref[valid].abs().mean())


# ------------------------------------------------------------------------------------------------
# prefill tile GEMM (gemm_prefill.hip): every epilogue vs an f32 reference of the same math
# ------------------------------------------------------------------------------------------------
@pytest.mark.parametrize("M,N_,K", [(1, 256, 64), (255, 512, 128), (257, 768, 4096), (1000, 256, 1088),
                                    (2304, 1024, 4096)])
def test_prefill_gemm_bf16(M, N_, K):
    from financial_chatbot_llm_amd.ops import gemm
    g = torch.Generator().manual_seed(M + N_)
    x, w = rnd(M, K, gen=g), rnd(N_, K, scale=0.05, gen=g)
    y = gemm.prefill_gemm(x.to(DEV), w.to(DEV))
    ref = x.float() @ w.float().t()
    close(y, ref, atol=2e-2 * ref.abs().max().item())
    assert y.shape == (M, N_) and y.dtype == torch.bfloat16


@pytest.mark.parametrize("M,epi", [(300, None), (2304, "residual"), (700, "slabs4")])
def test_prefill_gemm_production_down_shape_vs_fp32(M, epi):
    """The real Llama-3-8B down projection (N = 4096, K = 14336: 224 K-tiles, the tail split path at
    M = 300 and 700, a whole-tile round at 2304) against an fp32 reference computed on the GPU."""
    from financial_chatbot_llm_amd.ops import gemm
    g = torch.Generator(device=DEV).manual_seed(M)
    x = torch.randn((M, 14336), generator=g, device=DEV).to(torch.bfloat16)
    w = (torch.randn((4096, 14336), generator=g, device=DEV) * 0.02).to(torch.bfloat16)
    ref = x.float() @ w.float().t()
    if epi == "slabs4":
        P = gemm.prefill_gemm(x, w, "slabs", 4)
        close(P.sum(0), ref, atol=1e-3 * ref.abs().max().item(), rtol=1e-3)
        return
    if epi == "residual":
        r = torch.randn((M, 4096), generator=g, device=DEV).to(torch.bfloat16)
        y = gemm.prefill_gemm(x, w, "residual", residual=r)
        ref = ref + r.float()
    else:
        y = gemm.prefill_gemm(x, w)
    close(y, ref, atol=2e-2 * ref.abs().max().item())


@pytest.mark.parametrize("M", [300, 2304])
def test_prefill_gemm_production_gate_up_silu_vs_fp32(M):
    """The real gate|up + SiLU (N = 2 x 14336 = 28672 interleaved rows, K = 4096) against fp32."""
    from financial_chatbot_llm_amd.ops import gemm
    from financial_chatbot_llm_amd.ops.activation import silu_mul
    g = torch.Generator(device=DEV).manual_seed(M + 1)
    x = torch.randn((M, 4096), generator=g, device=DEV).to(torch.bfloat16)
    gate = (torch.randn((14336, 4096), generator=g, device=DEV) * 0.02).to(torch.bfloat16)
    up = (torch.randn((14336, 4096), generator=g, device=DEV) * 0.02).to(torch.bfloat16)
    w = gemm.interleave16(gate, up).contiguous()
    y = gemm.prefill_gemm(x, w, "silu")
    gf, uf = x.float() @ gate.float().t(), x.float() @ up.float().t()
    ref = torch.nn.functional.silu(gf) * uf
    close(y, ref, atol=2e-2 * ref.abs().max().item())


@pytest.mark.parametrize("M,S", [(37, 2), (600, 4), (513, 8)])
def test_prefill_gemm_split_k_slabs(M, S):
    from financial_chatbot_llm_amd.ops import gemm
    g = torch.Generator().manual_seed(S)
    N_, K = 512, 2048
    x, w = rnd(M, K, gen=g), rnd(N_, K, scale=0.05, gen=g)
    P = gemm.prefill_gemm(x.to(DEV), w.to(DEV), "slabs", S)
    assert P.shape == (S, M, N_) and P.dtype == torch.float32
    ref = torch.einsum("smk,snk->smn", x.float().view(M, S, K // S).transpose(0, 1),
                       w.float().view(N_, S, K // S).transpose(0, 1))
    close(P, ref, atol=1e-3 * ref.abs().max().item(), rtol=1e-3)     # f32 slabs: no bf16 rounding


def test_prefill_gemm_silu_and_residual_epilogues():
    from financial_chatbot_llm_amd.ops import gemm
    from financial_chatbot_llm_amd.ops.activation import silu_mul
    g = torch.Generator().manual_seed(5)
    M, F_, K = 300, 512, 1024
    x = rnd(M, K, gen=g)
    w = gemm.interleave16(rnd(F_, K, scale=0.05, gen=g), rnd(F_, K, scale=0.05, gen=g))
    y = gemm.prefill_gemm(x.to(DEV), w.to(DEV), "silu")
    ref = silu_mul((x.float() @ w.float().t()).to(torch.bfloat16), interleave16=True)
    close(y, ref, atol=2e-2 * ref.float().abs().max().item())
    r = rnd(M, 256, gen=g)
    w2 = rnd(256, K, scale=0.05, gen=g)
    y2 = gemm.prefill_gemm(x.to(DEV), w2.to(DEV), "residual", residual=r.to(DEV))
    ref2 = x.float() @ w2.float().t() + r.float()
    close(y2, ref2, atol=2e-2 * ref2.abs().max().item())


@pytest.mark.parametrize("M", [300, 700, 1300])
def test_prefill_gemm_fragment_tiled_weight(M):
    """The tile kernel reading the fragment-tiled weight (tile_weight, the decode kernels' layout) is
    bit-equal to the row-major form: bf16, SiLU, split-K slabs and the residual epilogue."""
    from financial_chatbot_llm_amd.ops import gemm
    g = torch.Generator().manual_seed(M)
    N_, K = 768, 1024
    x = rnd(M, K, gen=g).to(DEV)
    w = rnd(N_, K, scale=0.05, gen=g).to(DEV)
    wt = gemm.tile_weight(w)
    assert torch.equal(gemm.prefill_gemm_tiled(x, wt, N_), gemm.prefill_gemm(x, w))
    assert torch.equal(gemm.prefill_gemm_tiled(x, wt, N_, "silu"), gemm.prefill_gemm(x, w, "silu"))
    assert torch.equal(gemm.prefill_gemm_tiled(x, wt, N_, "slabs", 2), gemm.prefill_gemm(x, w, "slabs", 2))
    r = rnd(M, N_, gen=g).to(DEV)
    assert torch.equal(gemm.prefill_gemm_tiled(x, wt, N_, "residual", residual=r),
                       gemm.prefill_gemm(x, w, "residual", residual=r))
    close(gemm.prefill_gemm_tiled(x, wt, N_), x.float() @ w.float().t(), atol=2e-2)


@pytest.mark.parametrize("M,Hq,Hkv", [(1, 32, 8), (333, 32, 8), (1500, 8, 1)])
def test_prefill_qkv_rope_kv_write_fused(M, Hq, Hkv):
    """Fused QKV + RoPE + paged KV write == GEMM -> rope_kv_write (the unfused path), including
    tokens with no KV slot (slot -1) and llama3-scaled RoPE at large positions."""
    from financial_chatbot_llm_amd.ops import gemm
    from financial_chatbot_llm_amd.ops.attention import rope_cos_sin, rope_kv_write
    g = torch.Generator().manual_seed(M)
    D, K = 128, 1024
    x = rnd(M, K, gen=g).to(DEV)
    w = rnd((Hq + 2 * Hkv) * D, K, scale=0.03, gen=g).to(DEV)
    cs = rope_cos_sin(D, 8192, 500000.0, {"rope_type": "llama3", "factor": 8.0, "low_freq_factor": 1.0,
                                          "high_freq_factor": 4.0, "original_max_position_embeddings": 8192},
                      device=DEV)
    pos = torch.randint(0, 8192, (M,), generator=g, dtype=torch.int32).to(DEV)
    nb = (M + KV_BS - 1) // KV_BS + 1
    slots = torch.randperm(nb * KV_BS, generator=g)[:M].to(torch.int32)
    slots[::5] = -1
    slots = slots.to(DEV)
    kc = [torch.zeros((nb, Hkv, KV_BS * D), dtype=torch.bfloat16, device=DEV) for _ in range(2)]
    vc = [torch.zeros((nb, Hkv, KV_BS * D), dtype=torch.bfloat16, device=DEV) for _ in range(2)]
    q_ref = rope_kv_write((x.float() @ w.float().t()).to(torch.bfloat16), pos, cs, slots, kc[0], vc[0], Hq, Hkv, D)
    q = gemm.prefill_qkv_rope(x, w, pos, cs, slots, kc[1], vc[1], Hq, Hkv)
    scale = q_ref.float().abs().max().item()
    close(q, q_ref, atol=2e-2 * scale)
    close(kc[1], kc[0], atol=2e-2 * scale)
    close(vc[1], vc[0], atol=2e-2 * scale)
    # qscale: q leaves the epilogue times c before its one rounding; k / v untouched (bit-equal)
    c = 0.12753
    kc2, vc2 = torch.zeros_like(kc[1]), torch.zeros_like(vc[1])
    qc = gemm.prefill_qkv_rope(x, w, pos, cs, slots, kc2, vc2, Hq, Hkv, qscale=c)
    close(qc, q.float() * c, atol=1e-2 * scale * c)
    assert torch.equal(kc2, kc[1]) and torch.equal(vc2, vc[1])


@pytest.mark.parametrize("variant", [5, 7])
@pytest.mark.parametrize("Hq,Hkv,D,causal,lens,qscale", [
    (32, 8, 128, True, [(300, 1100), (17, 900), (70, 70), (130, 700)], 1.0),
    (32, 8, 128, True, [(257, 257), (64, 3000)], 12.0),      # peaky rows
    (8, 1, 128, True, [(40, 40), (33, 500)], 1.0),
])
def test_prefill_attention_prescaled_q(variant, Hq, Hkv, D, causal, lens, qscale, monkeypatch):
    """q handed over prescaled by scale * log2(e) at its ONE bf16 rounding (what the fused QKV epilogue
    does with qscale) on the prescaled-Q fold, with scale 1 / log2(e): as close to the fp32 reference
    as the exact-Q variant 5 fed bf16(q) -- the in-kernel prescale's second rounding (variant 6) is
    what costs precision on peaky rows -- plain and lean work lists."""
    monkeypatch.setattr(ops.attention, "LEAN_COST_GATE", False)
    g = torch.Generator().manual_seed(70)
    qlens = [a for a, _ in lens]
    ctx = [b for _, b in lens]
    tables, kc, vc = _paged_setup(ctx, Hkv, D, gen=g)
    cu = torch.tensor([0] + list(torch.tensor(qlens).cumsum(0)), dtype=torch.int32)
    qf = torch.randn(int(cu[-1]), Hq, D, generator=g) * qscale          # the rope output, f32
    ctx_t = torch.tensor(ctx, dtype=torch.int32)
    scale = 1 / math.sqrt(D)
    c = scale * 1.4426950408889634
    ref = ops.prefill(qf, cu, ctx_t, tables, kc, vc, scale, causal)
    q5 = qf.to(torch.bfloat16)
    qp = (qf * c).to(torch.bfloat16)
    args = (cu.to(DEV), ctx_t.to(DEV), tables.to(DEV), kc.to(DEV), vc.to(DEV))
    old = ops.attention.prefill_variant(5)
    try:
        out5 = ops.prefill(q5.to(DEV), *args, scale, causal, max_q_len=max(qlens))
        ops.attention.prefill_variant(variant)        # 7: the 32x32x16 kernel's prescaled-Q form
        outp = ops.prefill(qp.to(DEV), *args, 1 / 1.4426950408889634, causal, max_q_len=max(qlens), q_prescaled=True)
        wl = ops.attention.prefill_lean_list(cu.numpy(), ctx_t.numpy(), Hq // Hkv, Hkv, causal, cus=100000,
                                             min_chunk=1)
        outl = None
        if wl is not None:
            outl = ops.prefill(qp.to(DEV), *args, 1 / 1.4426950408889634, causal, max_q_len=max(qlens),
                               work=torch.from_numpy(wl).to(DEV), lean=(int(wl[0, 1]), int(wl[0, 2]), int(wl[0, 3])),
                               q_prescaled=True)
    finally:
        ops.attention.prefill_variant(old)
    e5 = (out5.float().cpu() - ref.float()).abs().max().item()
    ep = (outp.float().cpu() - ref.float()).abs().max().item()
    # on the peaky rows (qscale 12) the ONE rounding of q itself already costs variant 5 ~0.1 against
    # the f32-q reference; the prescaled form stays within 1.5x of that, and within 0.02 on typical rows
    assert ep <= 1.5 * e5 + 2e-3 and (qscale > 1 or ep <= 2e-2), (ep, e5)
    if outl is not None:
        assert (outl.float().cpu() - ref.float()).abs().max().item() <= 1.5 * e5 + 2e-2


@pytest.mark.parametrize("gelu", [False, True])
def test_prefill_gemm_bias_gelu_epilogue(gelu):
    """bge encoder projections: bf16(x @ w.T + b) [-> exact GELU] fused in the tile kernel."""
    from financial_chatbot_llm_amd.ops import gemm
    g = torch.Generator().manual_seed(11)
    M, N_, K = 1025, 768, 768
    x, w, b = rnd(M, K, gen=g), rnd(N_, K, scale=0.05, gen=g), rnd(N_, scale=0.5, gen=g)
    y = gemm.prefill_gemm(x.to(DEV), w.to(DEV), "bias_gelu" if gelu else "bias", bias=b.to(DEV))
    ref = x.float() @ w.float().t() + b.float()
    if gelu:
        ref = torch.nn.functional.gelu(ref)
    close(y, ref, atol=2e-2 * ref.abs().max().item())


def test_bge_encoder_bulk_tile_kernels_match_library_path(monkeypatch):
    """bge-base bulk batch (~24k tokens: the tile-kernel GEMMs with bias / GELU epilogues) vs the
    same weights through hipBLASLt + the separate GELU pass (PENNY_PREFILL_GEMM=0)."""
    from financial_chatbot_llm_amd.retrieval import BgeEmbedder
    emb = BgeEmbedder("bge-base-en", device=DEV)
    texts = [f"grocery purchase number {i} at store {i % 17} on the {i % 28 + 1}th" for i in range(2000)]
    a = emb.embed(texts).float().cpu()
    monkeypatch.setenv("PENNY_PREFILL_GEMM", "0")
    b = emb.embed(texts).float().cpu()
    cos = (a * b).sum(-1) / (a.norm(dim=-1) * b.norm(dim=-1))
    assert float(cos.min()) > 0.995, float(cos.min())


@pytest.mark.parametrize("T,E", [(300, 8), (2100, 8), (777, 4)])
def test_moe_prefill_fp8_tiles_matches_expert_loop(T, E):
    """Grouped fp8 tile GEMMs over device expert buckets (block-scaled 16x16x128 MFMA) == the
    per-expert fp8 x fp8 reference loop on the same quantized experts, with the intermediate
    rounded the way the tiles hand it over (MX blocks by default, per-row with PENNY_MOE_MX=0)."""
    from financial_chatbot_llm_amd.ops import gemm, moe
    g = torch.Generator(device=DEV).manual_seed(T)
    H, F_, K = 1024, 1536, 2
    w13 = (torch.randn((E, 2 * F_, H), device=DEV, generator=g) * 0.05).to(torch.bfloat16)
    w13 = torch.stack([gemm.interleave16(w13[e, :F_], w13[e, F_:]) for e in range(E)])
    q13, s13 = moe.quantize_fp8_rowwise(w13)
    w2 = (torch.randn((E, H, F_), device=DEV, generator=g) * 0.05).to(torch.bfloat16)
    q2, s2 = moe.quantize_fp8_rowwise(w2)
    h = torch.randn((T, H), device=DEV, generator=g).to(torch.bfloat16)
    logits = (torch.randn((T, E), device=DEV, generator=g) * 2).to(torch.bfloat16)
    if E == 4:                                   # an empty expert bucket
        logits[:, 3] = -30.0
    got = moe.moe_prefill_fp8_tiles(h, logits, q13.contiguous(), s13, q2.contiguous(), s2, K).float()
    # reference: dequantised experts in f32, the same per-row fp8 activation rounding
    topw, topi = moe.topk_softmax(logits, K)
    xq, xs = moe.quant_rows_fp8(h)
    xd = xq.float() * xs[:, None]
    ref = torch.zeros((T, H), device=DEV)
    for e in range(E):
        sel = (topi == e)
        rows = sel.any(1).nonzero().flatten()
        if rows.numel() == 0:
            continue
        w13d = q13[e].float() * s13[e][:, None]
        w2d = q2[e].float() * s2[e][:, None]
        a = gemm.silu_mul((xd[rows] @ w13d.t()).to(torch.bfloat16), interleave16=True)
        if moe.MX_HANDOFF:                       # the tiles hand the intermediate over in MX fp8
            y = moe._fake_quant_mx(a.float()) @ w2d.t()
        else:
            aq, as_ = moe.quant_rows_fp8(a)
            y = (aq.float() * as_[:, None]) @ w2d.t()
        wgt = (topw * sel).sum(1)[rows]
        ref[rows] += wgt[:, None] * y
    err = float((got - ref).abs().max() / ref.abs().max())
    assert err < 0.03, err


def test_mfma_scale_operand_map_dump():
    """Maps, for every (op_sel, lane, byte) of the B scale word, which accumulator entries it
    scales (one byte raised to 2^1 at a time) and writes the raw results to gpurun_out/ for the
    offline fit (diagnostic; asserts only that every experiment ran)."""
    from financial_chatbot_llm_amd.ops import _native as N
    from financial_chatbot_llm_amd.ops import moe
    g = torch.Generator().manual_seed(11)
    Am = torch.randint(1, 4, (16, 128), generator=g).float()
    Bm = torch.randint(1, 4, (16, 128), generator=g).float()
    def lanes(M):
        return torch.stack([M[l & 15, 32 * (l >> 4):32 * (l >> 4) + 32] for l in range(64)])
    Ad = lanes(Am).to(moe.FP8).view(torch.uint8).contiguous().view(torch.int32).to(DEV)
    Bd = lanes(Bm).to(moe.FP8).view(torch.uint8).contiguous().view(torch.int32).to(DEV)
    sad = torch.full((64,), 127, dtype=torch.int32, device=DEV)
    base_word = 127 | 127 << 8 | 127 << 16 | 127 << 24
    res = torch.zeros((4, 65, 4, 64, 4), dtype=torch.float32)
    for opsel in range(4):
        for lane in range(65):                 # lane 64: no change (baseline)
            for byte in range(4):
                sb = torch.full((64,), base_word, dtype=torch.int64)
                if lane < 64:
                    sb[lane] = base_word + (1 << (8 * byte))
                sbd = sb.to(torch.int32).to(DEV)
                out = torch.zeros(256, dtype=torch.float32, device=DEV)
                N.call("penny_probe_mfma_scale", N.ptr(Ad), N.ptr(Bd), N.ptr(sad), N.ptr(sbd), N.ptr(out), opsel,
                       N.stream())
                torch.cuda.synchronize()
                res[opsel, lane, byte] = out.cpu().view(64, 4)
    import os
    os.makedirs("gpurun_out", exist_ok=True)
    torch.save({"A": Am, "B": Bm, "res": res}, "gpurun_out/mfma_scale_probe.pt")
    assert torch.isfinite(res).all()


@pytest.mark.parametrize("opsel", [0, 1, 2, 3])
def test_mfma_scale_operand_semantics(opsel):
    """What the MX hand-off relies on in v_mfma_scale_f32_16x16x128_f8f6f4's B scale (measured with
    test_mfma_scale_operand_map_dump): byte `op_sel` of lane l's scale word scales column l & 15
    over the 16-element k chunks c of the fragment layout (lane l: row l & 15, chunks 2(l>>4),
    2(l>>4)+1) with moe.MX_CHUNK_BLOCK[c] == l >> 4 -- NOT the lane's own 32 elements."""
    import itertools
    from financial_chatbot_llm_amd.ops import _native as N
    from financial_chatbot_llm_amd.ops import moe
    g = torch.Generator().manual_seed(opsel)
    # small integers (exact in e4m3) for A [16 rows, 128 k] and B [16 rows, 128 k]
    Am = torch.randint(-3, 4, (16, 128), generator=g).float()
    Bm = torch.randint(-3, 4, (16, 128), generator=g).float()
    def lanes(M):   # lane l: row l & 15, k-block l >> 4 (32 bytes)
        return torch.stack([M[l & 15, 32 * (l >> 4):32 * (l >> 4) + 32] for l in range(64)])
    A8 = lanes(Am).to(moe.FP8).view(torch.uint8).contiguous().view(torch.int32)
    B8 = lanes(Bm).to(moe.FP8).view(torch.uint8).contiguous().view(torch.int32)
    sa = torch.full((64,), 127, dtype=torch.int32)
    sbytes = torch.randint(125, 130, (64, 4), generator=g, dtype=torch.int32)
    sb = (sbytes[:, 0] | sbytes[:, 1] << 8 | sbytes[:, 2] << 16 | sbytes[:, 3] << 24).to(torch.int32)
    out = torch.zeros(256, dtype=torch.float32, device=DEV)
    Ad, Bd, sad, sbd = A8.to(DEV), B8.to(DEV), sa.to(DEV), sb.to(DEV)      # alive across the launch
    N.call("penny_probe_mfma_scale", N.ptr(Ad), N.ptr(Bd), N.ptr(sad), N.ptr(sbd), N.ptr(out), opsel, N.stream())
    torch.cuda.synchronize()
    o = out.cpu().view(64, 4)
    C = torch.zeros(16, 16)
    for l in range(64):
        for r in range(4):
            C[4 * (l >> 4) + r, l & 15] = o[l, r]
    def model(byte):   # chunk c of column j scaled by byte `byte` of lane MX_CHUNK_BLOCK[c]*16 + j
        sc = torch.exp2((sbytes[:, byte].float() - 127)).view(4, 16)   # [block, j]
        ref = torch.zeros(16, 16)
        for c in range(8):
            ref += (Am[:, 16 * c:16 * c + 16] @ Bm[:, 16 * c:16 * c + 16].t()) * sc[moe.MX_CHUNK_BLOCK[c]][None, :]
        return ref
    fits = {b: float((model(b) - C).abs().max()) for b in range(4)}
    assert fits[opsel] == 0.0, fits


def _mx_setup(T=600, E=4, H=512, F_=512, seed=9):
    from financial_chatbot_llm_amd.ops import gemm, moe
    g = torch.Generator(device=DEV).manual_seed(seed)
    w13 = (torch.randn((E, 2 * F_, H), device=DEV, generator=g) * 0.05).to(torch.bfloat16)
    w13 = torch.stack([gemm.interleave16(w13[e, :F_], w13[e, F_:]) for e in range(E)])
    q13, s13 = moe.quantize_fp8_rowwise(w13)
    w2 = (torch.randn((E, H, F_), device=DEV, generator=g) * 0.05).to(torch.bfloat16)
    q2, s2 = moe.quantize_fp8_rowwise(w2)
    h = torch.randn((T, H), device=DEV, generator=g).to(torch.bfloat16)
    logits = (torch.randn((T, E), device=DEV, generator=g) * 2).to(torch.bfloat16)
    xq, xs, offsets, tok_idx, tok_w, inv = moe.route_quant_device(h, logits, 2, E)
    return q13.contiguous(), s13, q2.contiguous(), s2, xq, xs, offsets, tok_idx, tok_w, T * 2, E, H, F_


def _mx_scale_of(mxs, offsets, P, E, F_):
    """Decode the MX scale buffer into [P, F/128, 4] exponents (per K-tile and MFMA scale block)."""
    nkt = F_ // 128
    off = offsets.cpu().tolist()
    words = mxs.view(torch.uint8).cpu().view(-1, nkt, 4, 16, 4, 4)   # [tile][kt][wb][col][kblock][j]
    X = torch.zeros((P, nkt * 4), dtype=torch.int32)
    tm = 0
    for e in range(E):
        lo, hi = off[e], off[e + 1]
        for m0 in range(lo, hi, 256):
            for r in range(min(256, hi - m0)):
                wb, j, col = r // 64, (r % 64) // 16, r % 16
                X[m0 + r] = words[tm, :, wb, col, :, j].reshape(-1).to(torch.int32) - 127
            tm += 1
    return X


def test_moe_mx_gemm1_writes_fp8_and_block_scales():
    """GEMM1 of the MX hand-off alone: its e4m3 bytes x 2^X (X decoded from the scale layout) ==
    MX fp8 rounding of the bf16 SiLU intermediate the per-row pipeline's GEMM1 writes."""
    from financial_chatbot_llm_amd.ops import _native as N
    from financial_chatbot_llm_amd.ops import moe
    q13, s13, q2, s2, xq, xs, offsets, tok_idx, tok_w, P, E, H, F_ = _mx_setup()
    st = N.stream()
    a = torch.empty((P, F_), dtype=torch.bfloat16, device=DEV)
    N.call("penny_moe_gemm_prefill_fp8", N.ptr(xq), H, N.ptr(tok_idx), N.ptr(xs), N.ptr(offsets), N.ptr(q13),
           N.ptr(s13), None, N.ptr(a), F_, P, E, 2 * F_, H, 7, st)
    nkt = F_ // 128
    mxs = torch.zeros((((P + 255) // 256 + E) * nkt * 256,), dtype=torch.int32, device=DEV)
    aq = torch.zeros((P, F_), dtype=torch.uint8, device=DEV)
    N.call("penny_moe_gemm_prefill_fp8_mx", N.ptr(xq), H, N.ptr(tok_idx), N.ptr(xs), N.ptr(offsets), N.ptr(q13),
           N.ptr(s13), None, N.ptr(aq), F_, P, E, 2 * F_, H, 10, N.ptr(mxs), nkt, st)
    X = _mx_scale_of(mxs, offsets, P, E, F_).view(P, F_ // 128, 4)
    ref = moe._fake_quant_mx(a.float()).cpu()
    got = moe.mx_unblocks(moe.mx_blocks(aq.view(moe.FP8).float().cpu()) * torch.exp2(X.float())[..., None])
    amax = moe.mx_blocks(a.float().cpu()).abs().amax(-1)
    want_X = torch.where(amax > 0, torch.ceil(torch.log2(amax / 448.0)), torch.full_like(amax, -127.0))
    assert float((X.float() == want_X).float().mean()) > 0.999, (X[:2, :2], want_X[:2, :2])
    assert torch.allclose(got, ref, rtol=0, atol=1e-6 + 0.0), float((got - ref).abs().max())


def test_moe_mx_gemm2_applies_block_scales():
    """GEMM2 of the MX hand-off alone on a hand-built intermediate: unit scales (E8M0 127) ==
    the per-row GEMM2 at xs = 1; random scales == the fp32 reference of the scaled operand."""
    from financial_chatbot_llm_amd.ops import _native as N
    from financial_chatbot_llm_amd.ops import moe
    q13, s13, q2, s2, xq, xs, offsets, tok_idx, tok_w, P, E, H, F_ = _mx_setup()
    st = N.stream()
    g = torch.Generator(device=DEV).manual_seed(5)
    aq = (torch.randn((P, F_), device=DEV, generator=g) * 20).to(moe.FP8).view(torch.uint8)
    nkt = F_ // 128
    ntile = (P + 255) // 256 + E
    y_ref = torch.empty((P, H), dtype=torch.bfloat16, device=DEV)
    ones = torch.ones(P, dtype=torch.float32, device=DEV)
    N.call("penny_moe_gemm_prefill_fp8", N.ptr(aq), F_, None, N.ptr(ones), N.ptr(offsets), N.ptr(q2), N.ptr(s2),
           N.ptr(tok_w), N.ptr(y_ref), H, P, E, H, F_, 8, st)
    for mode in ("unit", "random"):
        if mode == "unit":
            mxs = torch.full((ntile * nkt * 1024,), 127, dtype=torch.uint8, device=DEV)
        else:
            mxs = torch.randint(124, 131, (ntile * nkt * 1024,), dtype=torch.uint8, device=DEV, generator=g)
        y = torch.empty((P, H), dtype=torch.bfloat16, device=DEV)
        N.call("penny_moe_gemm_prefill_fp8_mx", N.ptr(aq), F_, None, None, N.ptr(offsets), N.ptr(q2), N.ptr(s2),
               N.ptr(tok_w), N.ptr(y), H, P, E, H, F_, 11, N.ptr(mxs.view(torch.int32)), nkt, st)
        if mode == "unit":
            assert torch.equal(y, y_ref), float((y.float() - y_ref.float()).abs().max())
        else:
            X = _mx_scale_of(mxs.view(torch.int32), offsets, P, E, F_).to(DEV).view(P, F_ // 128, 4)
            xd = moe.mx_unblocks(moe.mx_blocks(aq.view(moe.FP8).float()) * torch.exp2(X.float())[..., None])
            off = offsets.cpu().tolist()
            ref = torch.zeros((P, H), device=DEV)
            for e in range(E):
                lo, hi = off[e], off[e + 1]
                ref[lo:hi] = (xd[lo:hi] @ (q2[e].float() * s2[e][:, None]).t()) * tok_w[lo:hi, None]
            err = float((y.float() - ref).abs().max() / ref.abs().max())
            assert err < 0.01, err


@pytest.mark.parametrize("T,E", [(1000, 8), (3001, 4)])
def test_moe_prefill_mx_handoff(T, E, monkeypatch):
    """MX hand-off of the fp8 tile pipeline (GEMM1 epilogue writes the SiLU intermediate as e4m3 +
    E8M0 scales per 32 columns, GEMM2 consumes them in its block-scaled MFMAs) vs the fp32
    per-expert reference with the same activation roundings (rows: per-row fp8; intermediate:
    MX fp8), and vs the per-row-quantised tile pipeline it replaces."""
    from financial_chatbot_llm_amd.ops import gemm, moe
    g = torch.Generator(device=DEV).manual_seed(T)
    H, F_, K = 1024, 1536, 2
    w13 = (torch.randn((E, 2 * F_, H), device=DEV, generator=g) * 0.05).to(torch.bfloat16)
    w13 = torch.stack([gemm.interleave16(w13[e, :F_], w13[e, F_:]) for e in range(E)])
    q13, s13 = moe.quantize_fp8_rowwise(w13)
    w2 = (torch.randn((E, H, F_), device=DEV, generator=g) * 0.05).to(torch.bfloat16)
    q2, s2 = moe.quantize_fp8_rowwise(w2)
    h = torch.randn((T, H), device=DEV, generator=g).to(torch.bfloat16)
    logits = (torch.randn((T, E), device=DEV, generator=g) * 2).to(torch.bfloat16)
    monkeypatch.setattr(moe, "MX_HANDOFF", False)
    rowq = moe.moe_prefill_fp8_tiles(h, logits, q13.contiguous(), s13, q2.contiguous(), s2, K).float()
    monkeypatch.setattr(moe, "MX_HANDOFF", True)
    got = moe.moe_prefill_fp8_tiles(h, logits, q13.contiguous(), s13, q2.contiguous(), s2, K).float()
    topw, topi = moe.topk_softmax(logits, K)
    xq, xs = moe.quant_rows_fp8(h)
    xd = xq.float() * xs[:, None]
    ref = torch.zeros((T, H), device=DEV)
    for e in range(E):
        sel = (topi == e)
        rows = sel.any(1).nonzero().flatten()
        if rows.numel() == 0:
            continue
        w13d = q13[e].float() * s13[e][:, None]
        w2d = q2[e].float() * s2[e][:, None]
        a = gemm.silu_mul((xd[rows] @ w13d.t()).to(torch.bfloat16), interleave16=True)
        y = moe._fake_quant_mx(a.float()) @ w2d.t()
        ref[rows] += (topw * sel).sum(1)[rows][:, None] * y
    err = (got - ref).abs()
    assert float(err.max() / ref.abs().max()) < 0.03, float(err.max() / ref.abs().max())
    # an activation on the other side of an e4m3 rounding boundary moves single outputs: bound
    # the mean (as the other fp8 pipeline tests do)
    assert float(err.mean()) < 0.01 * float(ref.abs().mean()) + 1e-4, (float(err.mean()), float(ref.abs().mean()))
    # accuracy: against the same pipeline with an UNquantised intermediate, the MX hand-off (scale
    # per 32 values) is no worse than the per-row quantisation it replaces
    exact = torch.zeros((T, H), device=DEV)
    for e in range(E):
        sel = (topi == e)
        rows = sel.any(1).nonzero().flatten()
        if rows.numel() == 0:
            continue
        w13d = q13[e].float() * s13[e][:, None]
        w2d = q2[e].float() * s2[e][:, None]
        a = gemm.silu_mul((xd[rows] @ w13d.t()).to(torch.bfloat16), interleave16=True).float()
        exact[rows] += (topw * sel).sum(1)[rows][:, None] * (a @ w2d.t())
    e_mx = float((got - exact).abs().mean())
    e_row = float((rowq - exact).abs().mean())
    assert e_mx <= 1.1 * e_row, (e_mx, e_row)


def test_moe_grouped_fp8_tiles_matches_reference():
    """Expert-parallel receive side on the tile kernel: y[i] = expert_{ids[i]}(x[i]) in the
    received (unsorted) row order, padding rows (id -1) zero."""
    from financial_chatbot_llm_amd.ops import gemm, moe
    g = torch.Generator(device=DEV).manual_seed(21)
    M, E, H, F_ = 700, 4, 1024, 1536
    w13 = (torch.randn((E, 2 * F_, H), device=DEV, generator=g) * 0.05).to(torch.bfloat16)
    w13 = torch.stack([gemm.interleave16(w13[e, :F_], w13[e, F_:]) for e in range(E)])
    q13, s13 = moe.quantize_fp8_rowwise(w13)
    w2 = (torch.randn((E, H, F_), device=DEV, generator=g) * 0.05).to(torch.bfloat16)
    q2, s2 = moe.quantize_fp8_rowwise(w2)
    x = torch.randn((M, H), device=DEV, generator=g).to(torch.bfloat16)
    ids = torch.randint(-1, E, (M,), device=DEV, generator=g, dtype=torch.int32)
    ids[ids == 2] = 1                                # an empty local expert
    got = moe.moe_grouped_fp8_tiles(x, ids, q13.contiguous(), s13, q2.contiguous(), s2).float()
    xq, xs = moe.quant_rows_fp8(x)
    xd = xq.float() * xs[:, None]
    ref = torch.zeros((M, H), device=DEV)
    for e in range(E):
        rows = (ids == e).nonzero().flatten()
        if rows.numel() == 0:
            continue
        a = gemm.silu_mul((xd[rows] @ (q13[e].float() * s13[e][:, None]).t()).to(torch.bfloat16), interleave16=True)
        aq, as_ = moe.quant_rows_fp8(a)
        ref[rows] = (aq.float() * as_[:, None]) @ (q2[e].float() * s2[e][:, None]).t()
    assert float(got[ids < 0].abs().max()) == 0.0
    err = float((got - ref).abs().max() / ref.abs().max())
    assert err < 0.03, err


def test_topp_threshold_is_bitwise_repeatable():
    """Integer (fixed-point) digit histograms: the top-p threshold of the same logits is bitwise
    identical across repeated launches and batch positions (float atomics made
    the nucleus edge depend on atomic ordering)."""
    from financial_chatbot_llm_amd.ops.sampling import topk_topp_threshold
    g = torch.Generator().manual_seed(5)
    V = 128256
    row = (torch.randn(1, V, generator=g) * 2.0).to(torch.bfloat16)
    lg = row.repeat(24, 1).to(DEV)
    t = torch.full((24,), 0.7, device=DEV)
    k = torch.zeros(24, dtype=torch.int32, device=DEV)
    p = torch.full((24,), 0.9, device=DEV)
    ths = [topk_topp_threshold(lg, t, k, p).cpu() for _ in range(20)]
    ref = ths[0][0]
    assert all(bool((th == ref).all()) for th in ths)


# ------------------------------------------------------------------------------------------------
# fused LM head + sampler (gemm_prefill.hip EPI_SAMPLE): no logits in HBM
# ------------------------------------------------------------------------------------------------
@pytest.mark.parametrize("M,V,K", [(1, 2048, 512), (37, 4096, 1024), (256, 2048, 512), (300, 1024, 256),
                                   (128, 128256, 4096)])
def test_fused_lm_head_sampler_matches_logits_then_sampler(M, V, K, monkeypatch):
    """Same tile accumulation as the bf16 tile GEMM -> identical bf16 logits -> the fused sample must
    equal ops.sample on those logits bit for bit (greedy and Gumbel rows); greedy rows also hold
    the fp32 reference's max logit up to bf16 rounding.  (The tile kernel at every M here: below
    128 rows ops.lm_head_sample takes the streaming kernel, tested below.)"""
    from financial_chatbot_llm_amd.ops import gemm
    monkeypatch.setenv("PENNY_LM_STREAM", "0")
    g = torch.Generator().manual_seed(M + V)
    x, w = rnd(M, K, gen=g).to(DEV), rnd(V, K, scale=0.05, gen=g).to(DEV)
    temps = torch.tensor([0.0 if i % 3 == 0 else (0.7 if i % 3 == 1 else 1.3) for i in range(M)], device=DEV)
    seeds = (torch.arange(M, dtype=torch.int64) * 7919 + 11).to(DEV)
    got = ops.lm_head_sample(x, w, temps, seeds)
    logits = gemm.prefill_gemm(x, w)
    want = ops.sample(logits, temps, seeds)
    assert torch.equal(got.cpu(), want.cpu())
    ref = (x.float() @ w.float().t())
    greedy = (temps <= 0).nonzero().flatten()
    picked = ref[greedy, got[greedy].long()]
    assert bool((picked >= ref[greedy].max(-1).values - 2e-2 * ref.abs().max()).all())
    # batch invariance: a row's sample does not depend on the other rows
    if M > 1:
        one = ops.lm_head_sample(x[1:2].contiguous(), w, temps[1:2].contiguous(), seeds[1:2].contiguous())
        assert int(one[0]) == int(got[1])


@pytest.mark.parametrize("M,V,K,nf,rowmajor,ring2", [(1, 2048, 512, 8, True, False), (37, 4096, 1024, 4, True, True),
                                                     (64, 4096, 1024, 8, False, False), (127, 2048, 512, 4, False, True),
                                                     (1, 128256, 4096, 8, True, False),
                                                     (100, 128256, 4096, 8, True, False)])
def test_lm_head_stream_sampler_matches_logits_then_sampler(M, V, K, nf, rowmajor, ring2):
    """Weight-streaming LM head + sampler (gemm_splitk.hip SK_SAMPLE, M <= 128): its accumulators are
    the SK_BF16 kernel's of the same shape -> identical bf16 logits -> the sample equals ops.sample
    on those logits bit for bit; the logits themselves match the fp32 reference; greedy rows pick
    the fp32 max up to bf16 rounding; a row's token does not depend on the other rows."""
    from financial_chatbot_llm_amd.ops import gemm
    g = torch.Generator().manual_seed(M * 3 + V)
    x, w = rnd(M, K, gen=g).to(DEV), rnd(V, K, scale=0.05, gen=g).to(DEV)
    wk = w if rowmajor else gemm.tile_weight(w)
    temps = torch.tensor([0.0 if i % 3 == 0 else (0.7 if i % 3 == 1 else 1.3) for i in range(M)], device=DEV)
    seeds = (torch.arange(M, dtype=torch.int64) * 7919 + 5).to(DEV)
    got = ops.lm_head_stream_sample(x, wk, temps, seeds, nf=nf, rowmajor=rowmajor, ring2=ring2)
    logits = gemm.splitk_bf16(x, wk, V, nf, rowmajor=rowmajor)
    ref = x.float() @ w.float().t()
    close(logits, ref, atol=3e-2)
    assert torch.equal(got.cpu(), ops.sample(logits, temps, seeds).cpu())
    greedy = (temps <= 0).nonzero().flatten()
    picked = ref[greedy, got[greedy].long()]
    assert bool((picked >= ref[greedy].max(-1).values - 2e-2 * ref.abs().max()).all())
    if M > 1:
        one = ops.lm_head_stream_sample(x[1:2].contiguous(), wk, temps[1:2].contiguous(), seeds[1:2].contiguous(),
                                        nf=nf, rowmajor=rowmajor, ring2=ring2)
        assert int(one[0]) == int(got[1])
    # the decode-size default route (ops.lm_head_sample below 128 rows) is this kernel
    if M <= 127 and V % 128 == 0:
        assert torch.equal(ops.lm_head_sample(x, w, temps, seeds).cpu(),
                           ops.sample(gemm.splitk_bf16(x, w, V, 8), temps, seeds).cpu())


@pytest.mark.parametrize("M", [1, 33, 127])
def test_lm_head_stream_vocab_shard_pairs(M):
    """Vocab-parallel form: a TP rank's padded LM-head shard (Llama-3 at TP=8: 16,032 rows in a
    16,128-row buffer) -> per-row (score, GLOBAL id) candidates equal to sample_shard over the same
    kernel's logits of the unpadded rows; padding rows never win."""
    from financial_chatbot_llm_amd.ops import gemm
    g = torch.Generator().manual_seed(M + 17)
    K, rows, Vpad, voff, vtot = 4096, 16032, 16128, 16032 * 3, 128256
    x = rnd(M, K, gen=g).to(DEV)
    wp = torch.zeros(Vpad, K, dtype=torch.bfloat16)
    wp[:rows] = rnd(rows, K, scale=0.05, gen=g)
    wp = wp.to(DEV)
    temps = torch.full((M,), 0.5, device=DEV)
    temps[::4] = 0.0
    seeds = (torch.arange(M, dtype=torch.int64) * 31 + 1).to(DEV)
    pairs = ops.lm_head_stream_sample(x, wp, temps, seeds, vvalid=rows, voff=voff, pairs=True)
    logits = gemm.splitk_bf16(x, wp, Vpad, 8)[:, :rows].contiguous()
    want = ops.sample_shard(logits, temps, seeds, voff, vtot)
    assert torch.equal(pairs.cpu(), want.cpu())
    assert bool(((pairs[:, 1] >= voff) & (pairs[:, 1] < voff + rows)).all())
    # the shard entry point routes decode sizes to the streaming kernel
    assert torch.equal(ops.lm_head_sample_shard(x, wp, rows, voff, temps, seeds).cpu(), pairs.cpu())


@pytest.mark.parametrize("M", [1, 37, 128, 256])
@pytest.mark.parametrize("N_,K,nf", [(8192, 1024, 2), (8192, 3584, 2), (8192, 3584, 4), (512, 1024, 8)])
def test_splitk_bf16_gemm_tp_row_shards(M, N_, K, nf):
    """bf16-output decode GEMM (SK_BF16, no K split) at the Llama-3-70B TP=8 row-parallel shard
    shapes (O [8192, 1024], down [8192, 3584]) vs the fp32 reference; row-major and tiled W agree
    bitwise; a strided X and a strided output are honoured."""
    from financial_chatbot_llm_amd.ops import gemm
    g = torch.Generator().manual_seed(M + N_ + K)
    x = rnd(M, K, gen=g).to(DEV)
    w = rnd(N_, K, scale=0.02, gen=g).to(DEV)
    y = gemm.splitk_bf16(x, w, N_, nf)
    close(y, x.float() @ w.float().t(), atol=3e-2)
    assert torch.equal(gemm.splitk_bf16(x, gemm.tile_weight(w), N_, nf, rowmajor=False), y)
    xw = torch.zeros(M, K + 64, dtype=torch.bfloat16, device=DEV)
    xw[:, 64:] = x
    out = torch.zeros(M, N_ + 8, dtype=torch.bfloat16, device=DEV)
    gemm.splitk_bf16(xw[:, 64:], w, N_, nf, out=out[:, :N_])
    assert torch.equal(out[:, :N_], y) and bool((out[:, N_:] == 0).all())


@pytest.mark.parametrize("M", [1, 64, 200])
def test_gateup_silu_nf2_tp8_shard(M):
    """The fused gate|up + SiLU kernel at nf = 2 on the Llama-3-70B TP=8 gate|up shard (interleave16
    of 2 x 3584 rows, K = 8192) vs the fp32 reference; row-major == tiled bitwise."""
    from financial_chatbot_llm_amd.ops import gemm
    g = torch.Generator().manual_seed(M + 2)
    Fr, K = 3584, 8192
    x = rnd(M, K, gen=g)
    gate, up = rnd(Fr, K, scale=0.02, gen=g), rnd(Fr, K, scale=0.02, gen=g)
    wi = gemm.interleave16(gate, up).to(DEV).contiguous()
    y = gemm.gateup_silu(x.to(DEV), wi, 2 * Fr, 2, rowmajor=True)
    assert torch.equal(gemm.gateup_silu(x.to(DEV), gemm.tile_weight(wi), 2 * Fr, 2), y)
    xd = x.to(DEV).float()
    gf, uf = xd @ gate.to(DEV).float().t(), xd @ up.to(DEV).float().t()
    close(y, torch.nn.functional.silu(gf) * uf, atol=3e-2)


@pytest.mark.parametrize("M,S,nf", [(1, 8, 4), (64, 4, 2), (160, 2, 8)])
def test_gateup_splitk_reduce_silu_tp8_shard(M, S, nf):
    """Split-K gate|up (slabs + the reduce-SiLU pass) on the Llama-3-70B TP=8 gate|up shard vs the
    fp32 reference; row-major == tiled bitwise; the reduce pass equals silu_mul over the summed slabs."""
    from financial_chatbot_llm_amd.ops import gemm
    from financial_chatbot_llm_amd.ops.activation import silu_mul
    g = torch.Generator().manual_seed(M + 7)
    Fr, K = 3584, 8192
    x = rnd(M, K, gen=g)
    gate, up = rnd(Fr, K, scale=0.02, gen=g), rnd(Fr, K, scale=0.02, gen=g)
    wi = gemm.interleave16(gate, up).to(DEV).contiguous()
    y = gemm.gateup_splitk(x.to(DEV), wi, 2 * Fr, S, nf, rowmajor=True)
    assert torch.equal(gemm.gateup_splitk(x.to(DEV), gemm.tile_weight(wi), 2 * Fr, S, nf), y)
    P = gemm.splitk_partials(x.to(DEV), wi, 2 * Fr, S, nf, rowmajor=True)
    assert torch.equal(silu_mul(P.sum(0).to(torch.bfloat16), interleave16=True), y)
    xd = x.to(DEV).float()
    gf, uf = xd @ gate.to(DEV).float().t(), xd @ up.to(DEV).float().t()
    close(y, torch.nn.functional.silu(gf) * uf, atol=3e-2)


@pytest.mark.parametrize("Vs", [16033, 1001])
def test_sample_shard_any_width(Vs):
    """a vocab shard whose width is not a multiple of 8 (row stride V/tp) samples on the
    device (an aligned copy) instead of asserting; greedy rows equal the argmax, and the result
    equals the aligned-buffer call bit for bit."""
    g = torch.Generator().manual_seed(Vs)
    B = 9
    logits = rnd(B, Vs, gen=g).to(DEV)
    temps = torch.full((B,), 0.8, device=DEV)
    temps[::3] = 0.0
    seeds = (torch.arange(B, dtype=torch.int64) + 3).to(DEV)
    pairs = ops.sample_shard(logits, temps, seeds, 5 * Vs, 8 * Vs)
    buf = torch.zeros(B, Vs + 8 - Vs % 8, dtype=torch.bfloat16, device=DEV)
    buf[:, :Vs] = logits
    assert torch.equal(pairs.cpu(), ops.sample_shard(buf[:, :Vs], temps, seeds, 5 * Vs, 8 * Vs).cpu())
    greedy = (temps <= 0).nonzero().flatten()
    assert torch.equal(pairs[greedy, 1].cpu().long() - 5 * Vs, logits[greedy].float().argmax(-1).cpu())
    assert ops.sample(logits, temps, seeds).shape == (B,)


@pytest.mark.parametrize("M", [127, 128])
def test_fused_vs_unfused_sampling_token_agreement(M):
    """the fused LM-head sampler (tile GEMM, from 128 rows) and hipBLASLt logits + the
    sampler accumulate the logits in different orders, so the same seed can pick a different token
    when two candidates' scores are within logit rounding.  Llama-3-8B LM-head shape: the rate is
    measured (printed) and must stay rare; tokens are reproducible only up to logit rounding."""
    g = torch.Generator(device=DEV).manual_seed(11)
    w = (torch.randn((128256, 4096), generator=g, device=DEV) * 0.02).to(torch.bfloat16)
    h = torch.randn((M, 4096), generator=g, device=DEV).to(torch.bfloat16)
    temps = torch.full((M,), 0.5, device=DEV)
    temps[::5] = 0.0
    seeds = torch.arange(M, dtype=torch.int64, device=DEV) * 7919 + 3
    fused = ops.lm_head_sample(h, w, temps, seeds)
    unfused = ops.sample(torch.nn.functional.linear(h, w), temps, seeds)
    agree = float((fused == unfused).float().mean())
    print(f"fused vs unfused sampling agreement at M={M}: {agree:.4f}")
    assert agree >= 0.95


def test_fused_lm_head_graph_decode_falls_back_for_top_p(monkeypatch):
    """A hipGraph decode bucket captured with the fused sampler still honours top-k / top-p rows
    (those steps run eagerly through the logits + filtered sampler)."""
    monkeypatch.setenv("PENNY_FUSED_LM_HEAD", "force")
    from financial_chatbot_llm_amd.config import EngineConfig
    from financial_chatbot_llm_amd.engine import LLMEngine, SamplingParams
    cfg = EngineConfig(model="llama-tiny", device="cuda", num_kv_blocks=64, max_model_len=1024,
                       max_num_seqs=4, graph_batch_sizes=(1, 2, 4))
    eng = LLMEngine(cfg)
    eng.warmup()
    prompts = [list(range(100, 160)), list(range(7, 30))]
    greedy = eng.generate(prompts, SamplingParams(temperature=0.0, max_tokens=6, ignore_eos=True))
    assert eng.runner.stats.get("fused_lm_head_steps", 0) > 0 or any(G.fused for G in eng.runner.graphs.values())
    filt = eng.generate(prompts, SamplingParams(temperature=0.8, top_p=0.5, top_k=5, max_tokens=6, ignore_eos=True,
                                                seed=3))
    assert all(len(o) == 6 for o in greedy + filt)
    monkeypatch.setenv("PENNY_FUSED_LM_HEAD", "0")
    eng2 = LLMEngine(cfg)
    eng2.warmup()
    # filtered rows take the unfused sampler on both engines (eager fallback vs the unfused graph)
    assert eng2.generate(prompts, SamplingParams(temperature=0.8, top_p=0.5, top_k=5, max_tokens=6,
                                                 ignore_eos=True, seed=3)) == filt


@pytest.mark.parametrize("M,N_,K,epi", [(512, 6144, 4096, None), (2560, 1024, 2048, "silu"), (300, 512, 1024, "residual"),
                                        (1000, 768, 768, "bias_gelu"),
                                        # production shapes around the tail's decision points
                                        (2304, 4096, 4096, None), (2304, 4096, 14336, "residual"),
                                        (768, 6144, 4096, None), (1024, 28672, 4096, "silu"),
                                        (4608, 4096, 4096, "residual")])
def test_prefill_gemm_wave_quantisation_tail(M, N_, K, epi, monkeypatch):
    """Tail tiles split along K over idle CUs (last split combines in registers) equal the whole-tile
    launch up to f32 summation order, every call (the ticket counters reset themselves)."""
    from financial_chatbot_llm_amd.ops import gemm
    g = torch.Generator().manual_seed(M + N_)
    x, w = rnd(M, K, gen=g).to(DEV), rnd(N_, K, scale=0.05, gen=g).to(DEV)
    kw = {}
    if epi == "residual":
        kw["residual"] = rnd(M, N_, gen=g).to(DEV)
    if epi == "bias_gelu":
        kw["bias"] = rnd(N_, gen=g).to(DEV)
    monkeypatch.setenv("PENNY_GEMM_TAIL", "0")
    whole = gemm.prefill_gemm(x, w, epi, **kw)
    monkeypatch.setenv("PENNY_GEMM_TAIL", "1")
    outs = [gemm.prefill_gemm(x, w, epi, **kw) for _ in range(3)]
    for y in outs:
        close(y, whole, atol=1e-2 * whole.float().abs().max().item())
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[1], outs[2])


@pytest.mark.parametrize("D", [64, 128])
def test_rope_qk_matches_reference(D):
    """Context-parallel RoPE (penny_rope_qk): rotated q and k heads at arbitrary (zig-zag) positions,
    no cache write, vs the fp32 reference."""
    from financial_chatbot_llm_amd.ops.attention import _rope_ref, rope_cos_sin, rope_qk
    g = torch.Generator().manual_seed(D)
    T, Hq, Hkv = 300, 8, 2
    qkv = rnd(T, (Hq + 2 * Hkv) * D, gen=g)
    pos = torch.randperm(4096, generator=g)[:T].to(torch.int32)
    cs = rope_cos_sin(D, 4096, 500000.0)
    got = rope_qk(qkv.to(DEV), pos.to(DEV), cs.to(DEV), Hq, Hkv, D)
    ref = _rope_ref(qkv.view(T, -1, D)[:, :Hq + Hkv].float(), pos, cs)
    assert got.shape == (T, Hq + Hkv, D)
    close(got, ref, atol=2e-2)


# ---- 128 x 128 tile kernel (gemm_mid.hip): the Llama-3-70B TP=8 shard shapes ----
@pytest.mark.parametrize("variant", [0, 1, 2])
@pytest.mark.parametrize("name,M,S", [("qkv", 384, 4), ("qkv", 1000, 1), ("o", 300, 1), ("o", 1536, 2),
                                       ("gate_up", 513, 1), ("gate_up", 384, 2), ("down", 257, 1), ("down", 768, 2)])
def test_mid_gemm_tp8_shard_shapes_vs_fp32(variant, name, M, S):
    """Every epilogue form of the mid tile kernel at the 70B TP=8 shards against fp32 on the GPU:
    QKV (1280 x 8192) slabs for the RoPE pass, O (8192 x 1024) and down (8192 x 3584) bf16 for the
    all-reduce (S > 1: slabs + penny_splitk_reduce), gate|up (7168 x 8192 interleave16) + SiLU (S > 1:
    slabs + reduce-SiLU); M not a multiple of the 128-row tile included."""
    from financial_chatbot_llm_amd.ops import gemm
    N_, K = {"qkv": (1280, 8192), "o": (8192, 1024), "gate_up": (7168, 8192), "down": (8192, 3584)}[name]
    old = gemm.mid_variant(variant)
    try:
        _mid_case(gemm, name, M, S, N_, K)
    finally:
        gemm.mid_variant(old)


def _mid_case(gemm, name, M, S, N_, K):
    g = torch.Generator(device=DEV).manual_seed(M * 7 + S)
    x = torch.randn((M, K), generator=g, device=DEV).to(torch.bfloat16)
    w = (torch.randn((N_, K), generator=g, device=DEV) * 0.02).to(torch.bfloat16)
    ref = x.float() @ w.float().t()
    if name == "gate_up":
        y = gemm.mid_linear(x, w, S, "silu")
        gt = ref.to(torch.bfloat16).float().view(M, N_ // 32, 2, 16)
        ref = (torch.nn.functional.silu(gt[:, :, 0]) * gt[:, :, 1]).reshape(M, N_ // 2)
        assert y.shape == (M, N_ // 2)
        close(y, ref, atol=2e-2 * ref.abs().max().item())
        return
    if name == "qkv" and S > 1:
        out = gemm.mid_linear(x, w, S, None, slabs=True)
        assert isinstance(out, gemm.Slabs) and out.P.shape == (S, M, N_)
        close(out.P.sum(0), ref, atol=1e-3 * ref.abs().max().item(), rtol=1e-3)
        return
    y = gemm.mid_linear(x, w, S)
    assert y.shape == (M, N_) and y.dtype == torch.bfloat16
    close(y, ref, atol=2e-2 * ref.abs().max().item())


@pytest.mark.parametrize("N_,K,M,S", [(4096, 4096, 320, 4), (4096, 4096, 700, 2), (4096, 14336, 384, 4)])
def test_linear_8b_small_prefill_steps_take_mid_slabs(N_, K, M, S):
    """Llama-3-8B O / down at small prefill steps through ``linear`` (the production call, slabs for
    the add&RMSNorm consumer): the policy's 128 x 128 tile slabs, equal to the fp32 product."""
    from financial_chatbot_llm_amd.ops import gemm
    assert gemm.prefill_choice(M, N_, K, None, True, fused_residual=True) == f"M{S}"
    g = torch.Generator(device=DEV).manual_seed(M)
    x = torch.randn((M, K), generator=g, device=DEV).to(torch.bfloat16)
    w = (torch.randn((N_, K), generator=g, device=DEV) * 0.02).to(torch.bfloat16)
    r = torch.randn((M, N_), generator=g, device=DEV).to(torch.bfloat16)
    out = gemm.linear(x, w, slabs=True, fuse_residual=r)
    assert isinstance(out, gemm.Slabs) and out.P.shape == (S, M, N_)
    ref = x.float() @ w.float().t()
    close(out.P.sum(0), ref, atol=1e-3 * ref.abs().max().item(), rtol=1e-3)


def test_mid_gemm_residual_epilogue_and_slab_exactness():
    """Residual epilogue (bf16(acc) + R, like GEMM-then-add) and split-K slabs equal to the f32
    per-slice products."""
    from financial_chatbot_llm_amd.ops import gemm
    g = torch.Generator().manual_seed(11)
    M, N_, K, S = 200, 384, 1024, 4
    x, w, r = rnd(M, K, gen=g), rnd(N_, K, scale=0.05, gen=g), rnd(M, N_, gen=g)
    y = gemm.mid_gemm(x.to(DEV), w.to(DEV), "residual", residual=r.to(DEV))
    ref = (x.float() @ w.float().t()).to(torch.bfloat16).float() + r.float()
    close(y, ref, atol=2e-2 * ref.abs().max().item())
    P = gemm.mid_gemm(x.to(DEV), w.to(DEV), "slabs", S)
    refP = torch.einsum("smk,snk->smn", x.float().view(M, S, K // S).transpose(0, 1),
                        w.float().view(N_, S, K // S).transpose(0, 1))
    close(P, refP, atol=1e-3 * refP.abs().max().item(), rtol=1e-3)


@pytest.mark.parametrize("T,E,H,K", [(1, 8, 8, 2), (48, 8, 4096, 2), (65, 9, 520, 4), (512, 16, 2048, 8), (3, 4, 16384, 1), (7, 3, 10248, 3)])
def test_moe_decode_route(T, E, H, K):
    """Router, choice, quantised rows and buckets in one launch: the choice of its own bf16 logits, in buckets that hold every pair once."""
    from financial_chatbot_llm_amd.ops import _native as N, moe
    g = torch.Generator().manual_seed(T + E)
    h, router = rnd(T, H, gen=g), rnd(E, H, scale=H ** -0.5, gen=g)
    x, rw = h.to(DEV), router.to(DEV)
    ws = moe.MoEWorkspace(max(T, 8), K, E, H, 16, DEV)
    z = h.double() @ router.double().t()
    for _ in range(2):                                                   # the ticket is back at zero
        N.call("penny_moe_decode_route", N.ptr(x), H, N.ptr(rw), T, H, E, K, N.ptr(ws.xq), N.ptr(ws.xs), N.ptr(ws.pairs[0]),
               N.ptr(ws.pairs[1]), N.ptr(ws.ticket), N.ptr(ws.sorted_tok), N.ptr(ws.sorted_w), N.ptr(ws.offsets), N.ptr(ws.inv), N.stream())
        q, s = moe.quant_rows_fp8(x)
        assert torch.equal(ws.xq[:T], q.view(torch.uint8)) and torch.equal(ws.xs[:T], s)
        idx, w = ws.pairs[0].flatten()[:T * K].view(T, K).cpu().long(), ws.pairs[1].flatten().view(torch.float32)[:T * K].view(T, K).cpu()
        assert all(len(set(r.tolist())) == K for r in idx) and int(idx.min()) >= 0 and int(idx.max()) < E
        # chosen logits within one bf16 step (2^-8 of the largest either way) of the best ones, in order
        best = z.sort(1, descending=True).values[:, :K]
        tol = 2 ** -7 * z.abs().amax(1, keepdim=True) + 1e-6
        assert ((z.gather(1, idx) - best).abs() <= tol).all()
        want = torch.softmax(z.gather(1, idx), 1)
        assert ((w - want).abs() <= 2 * tol).all() and torch.allclose(w.sum(1), torch.ones(T), atol=1e-5)
        off, inv = ws.offsets.cpu().tolist(), ws.inv[:T * K].cpu().long()
        assert off[0] == 0 and off[-1] == T * K and sorted(inv.tolist()) == list(range(T * K))
        flat = idx.flatten()
        assert all(off[e] <= p < off[e + 1] for p, e in zip(inv.tolist(), flat.tolist()))
        assert torch.equal(ws.sorted_tok.cpu().long()[inv], torch.arange(T * K) // K)
        assert torch.equal(ws.sorted_w.cpu()[inv], w.flatten())


@pytest.mark.parametrize("n", [8, 2040, 2056, 4104, 16384, 16392, 40000])
def test_quant_rows_sizes(n):
    """Rows around what a thread holds in one, two, four and eight pieces, and longer ones: scale amax / 448, values the nearest e4m3."""
    from financial_chatbot_llm_amd.ops import moe
    x = (torch.randn(3, n + 8, generator=torch.Generator().manual_seed(n)) * 3).to(torch.bfloat16)[:, :n]
    x[2] = 0
    q, s = moe.quant_rows_fp8(x.to(DEV))
    amax = x.float().abs().amax(1)
    assert torch.equal(s.cpu(), torch.where(amax > 0, amax / 448.0, torch.ones(3)))
    y, got = x.float() * (1.0 / s.cpu())[:, None], q.cpu().float()
    # half a step of e4m3: 3 mantissa bits, 2^-10 below 2^-6
    assert ((got - y).abs() <= y.abs().clamp(min=2.0 ** -6) * 2.0 ** -4 + 1e-6).all()
