"""Filtered top-k: candidate counts around the ranking's and the sort's limits, several calls through one workspace, ties and
scores that are not numbers, corpus sizes around a block's share."""
import pytest
import torch

from financial_chatbot_llm_amd import ops

pytestmark = pytest.mark.gpu


def corpus(sizes, N, D, seed):
    """N rows; user u + 1 owns sizes[u] of them, the rest belong to user 0."""
    g = torch.Generator().manual_seed(seed)
    users = torch.zeros(N, dtype=torch.int32)
    perm, o = torch.randperm(N, generator=g), 0
    for u, n in enumerate(sizes):
        users[perm[o:o + n]] = u + 1
        o += n
    x = torch.randint(-3, 4, (N, D), generator=g).to(torch.bfloat16)      # whole numbers: exact sums, many ties
    dates = torch.randint(0, 1000, (N,), generator=g)
    q = torch.randint(-3, 4, (len(sizes) + 1, D), generator=g).to(torch.bfloat16)
    return x, users, dates, q


@pytest.mark.parametrize("sizes,N,D", [([0, 1, 2], 3, 8), ([5, 255, 256, 257, 300], 1100, 64), ([1024, 1, 700, 8192], 12000, 64),
                                       ([9000], 9001, 8), ([100] * 40, 4097, 768)])
def test_sizes(sizes, N, D):
    x, users, dates, q = corpus(sizes, N, D, len(sizes))
    nq, kmax = len(sizes) + 1, 300
    who = torch.tensor([u + 1 for u in range(len(sizes))] + [len(sizes) + 5], dtype=torch.int32)
    dev = [t.cuda() for t in (x, users, dates, q, who)]
    for since, k in ((0, kmax), (500, 10), (0, 1)):
        floor, ks = torch.full((nq,), since, dtype=torch.int64), torch.full((nq,), k, dtype=torch.int32)
        got = ops.filtered_topk(*dev, floor.cuda(), ks.cuda(), kmax)
        want = ops.filtered_topk(x, users, dates, q, who, floor, ks, kmax)
        assert torch.equal(got[2].cpu(), want[2]) and torch.equal(got[1].cpu(), want[1])
        small = torch.tensor([n <= 8192 for n in sizes] + [True])          # the library's top-k breaks ties its own way
        assert torch.equal(got[0].cpu()[small], want[0][small])


@pytest.mark.parametrize("D", [8, 520, 1024])
@pytest.mark.parametrize("nq", [1, 3, 17, 64])
def test_one_block_and_several(nq, D):
    """Counts around what one block ranks alone, and more queries than a block each: contiguous rows of a user, which hit whole waves."""
    sizes = ([128, 129, 127, 2, 1000, 257] * 11)[:nq]
    x, users, dates, q = corpus(sizes, sum(sizes) + 600, D, nq + D)
    users = users.sort().values
    who, ks = torch.arange(1, nq + 1, dtype=torch.int32), torch.full((nq,), 200, dtype=torch.int32)
    for since in (0, 400):
        floor = torch.full((nq,), since, dtype=torch.int64)
        want = ops.filtered_topk(x, users, dates, q[:nq], who, floor, ks, 260)
        for _ in range(2):                                                 # the counters are back at zero
            got = ops.filtered_topk(*(t.cuda() for t in (x, users, dates, q[:nq], who, floor, ks)), 260)
            for g, w in zip(got, want):
                assert torch.equal(g.cpu(), w)


def test_not_a_number():
    x, users, dates, q = corpus([200], 300, 64, 7)
    x[users.nonzero().flatten()[:3]] = float("nan")
    ids, _, count = ops.filtered_topk(x.cuda(), users.cuda(), dates.cuda(), q[:1].cuda(), torch.tensor([1]).cuda(),
                                      torch.tensor([0]).cuda(), torch.tensor([200]).cuda(), 200)
    assert int(count[0]) == 200 and set(ids[0].tolist()) == set(users.nonzero().flatten().tolist())


def test_workspaces(monkeypatch):
    """Batches of several sizes share a set of lists, threads do not, and one whose call failed is not used again."""
    import threading

    from financial_chatbot_llm_amd.ops import retrieval
    sizes = [5, 300, 40, 700, 1, 90]
    x, users, dates, q = corpus(sizes, 3000, 64, 11)
    who, floor, ks = torch.arange(1, 7, dtype=torch.int32), torch.zeros(6, dtype=torch.int64), torch.full((6,), 50, dtype=torch.int32)
    rows, rest = [t.cuda() for t in (x, users, dates)], [t.cuda() for t in (q[:6], who, floor, ks)]
    want = ops.filtered_topk(x, users, dates, q[:6], who, floor, ks, 50)
    made, zeros = [], torch.zeros

    def counted(*a, **k):
        made.append(zeros(*a, **k))
        return made[-1]

    def check(n):
        for g, w in zip(ops.filtered_topk(*rows, *(t[:n] for t in rest), 50), want):
            assert torch.equal(g.cpu(), w[:n])

    monkeypatch.setattr(retrieval, "_FREE", [])
    monkeypatch.setattr(torch, "zeros", counted)
    check(6)
    for n in (1, 5, 2, 6, 3):
        check(n)
    assert len(made) == 1                                  # one set, made by the first call
    call = retrieval.N.call

    def fails(name, *args):                                # behind the filter: the counters are not back at zero
        made[-1].fill_(2)
        torch.cuda.synchronize()
        raise RuntimeError(name)

    monkeypatch.setattr(retrieval.N, "call", fails)
    with pytest.raises(RuntimeError):
        check(6)
    monkeypatch.setattr(retrieval.N, "call", call)
    check(6)
    assert len(made) == 2
    errors = []

    def worker():
        try:
            for n in (2, 6, 4) * 5:
                check(n)
        except BaseException as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=worker) for _ in range(12)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors and len(retrieval._FREE) <= 8


def test_calls_in_a_row():
    """Calls behind one another, whose lists, counters and counts for the host are one set, with rows ranked alone, by several blocks, by
    sorting and on the host's side."""
    sizes = [90, 200, 1500, 9000, 0, 3]
    x, users, dates, q = corpus(sizes, 14000, 64, 11)
    rows = [t.cuda() for t in (x, users, dates)]
    calls = []
    for i in range(24):
        pick = [(i + j) % 6 for j in range(1 + i % 5)]
        if i % 3:                                                          # most calls without a wait of their own
            pick = [u for u in pick if u != 3] or [0]
        who = torch.tensor([u + 1 for u in pick], dtype=torch.int32)
        floor, ks = torch.full((len(pick),), 13 * i), torch.full((len(pick),), 40 + i, dtype=torch.int32)
        calls.append((q[pick], who, floor, ks, [u != 3 for u in pick]))
    dev = [[t.cuda() for t in c[:4]] for c in calls]
    torch.cuda.synchronize()
    got = [ops.filtered_topk(*rows, *c, 64) for c in dev]
    for c, (ids, scores, counts) in zip(calls, got):
        want = ops.filtered_topk(x, users, dates, *c[:4], 64)
        assert torch.equal(counts.cpu(), want[2]) and torch.equal(scores.cpu(), want[1])
        assert torch.equal(ids.cpu()[c[4]], want[0][c[4]])


@pytest.mark.parametrize("before", [0, 40])
def test_results_are_complete_on_return(before):
    """Nothing of a call is left on its stream when it returns, also behind a few milliseconds of other work: another stream may read its
    results at once."""
    sizes = [4000] * 16 + [90, 0, 200]
    x, users, dates, q = corpus(sizes, sum(sizes) + 50, 256, 5)
    nq, other, own = len(sizes), torch.cuda.Stream(), torch.cuda.Stream()
    who, floor, ks = torch.arange(1, nq + 1, dtype=torch.int32), torch.zeros(nq, dtype=torch.int64), torch.full((nq,), 300, dtype=torch.int32)
    dev = [t.cuda() for t in (x, users, dates, q[:nq], who, floor, ks)]
    want = ops.filtered_topk(x, users, dates, q[:nq], who, floor, ks, 300)
    busy = torch.randn((4096, 4096), device="cuda")
    torch.cuda.synchronize()
    for _ in range(3):
        with torch.cuda.stream(own):
            for _ in range(before):
                busy @ busy
            got = ops.filtered_topk(*dev, 300)
            assert own.query()
        with torch.cuda.stream(other):
            for g, w in zip(got, want):
                assert torch.equal(g.cpu(), w)
        torch.cuda.synchronize()
