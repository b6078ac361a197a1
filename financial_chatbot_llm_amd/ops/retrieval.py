"""K15: filtered exact top-k over an HBM-resident corpus (user_id == u AND date >= t)."""
from __future__ import annotations

import threading
from typing import List, Tuple

import torch

from . import _native as N

SORT_CAP = 8192


def filtered_topk_ref(corpus, user_codes, dates, queries, q_user, q_floor, ks, kmax):
    nq = queries.shape[0]
    ids = torch.full((nq, kmax), -1, dtype=torch.int32, device=corpus.device)
    scores = torch.zeros((nq, kmax), dtype=torch.float32, device=corpus.device)
    counts = torch.zeros((nq,), dtype=torch.int32, device=corpus.device)
    for i in range(nq):
        mask = (user_codes == q_user[i]) & (dates >= q_floor[i])
        rows = torch.nonzero(mask).flatten()
        if rows.numel() == 0:
            continue
        s = corpus[rows].float() @ queries[i].float()
        # descending score, ties by smaller row id (rows are ascending -> stable sort)
        order = torch.sort(-s, stable=True).indices
        k = min(int(ks[i]), rows.numel(), kmax)
        ids[i, :k] = rows[order[:k]].to(torch.int32)
        scores[i, :k] = s[order[:k]]
        counts[i] = k
    return ids, scores, counts


# Candidate lists that no call holds: (device, stream, set), at most eight, the longest unused dropped first.  A set serves the
# calls of one stream, whatever their sizes; a call takes one (or makes it), so two threads never share it, and hands it back
# when its kernels have left the counters at zero again -- a call that fails does not.
_Set = Tuple[torch.Tensor, torch.Tensor, torch.Tensor, torch.Tensor]
_FREE: List[Tuple[int, int, _Set]] = []
_LOCK = threading.Lock()
_KEEP = 8


def _take(n: int, device: torch.device, stream: int) -> _Set:
    """Counters [64, 32] of zeros, rows and scores of at least ``n`` candidates, 64 result counts in pinned host memory."""
    with _LOCK:
        for i, (d, s, ws) in enumerate(_FREE):
            if d == device.index and s == stream and ws[1].numel() >= n:
                return _FREE.pop(i)[2]
    n = 1 << (n - 1).bit_length()          # few sizes: a smaller call fits behind a larger one
    return (torch.zeros((64, 32), dtype=torch.int32, device=device), torch.empty(n, dtype=torch.int32, device=device),
            torch.empty(n, dtype=torch.float32, device=device), torch.empty(64, dtype=torch.int32, pin_memory=True))


def _hand_back(ws: _Set, device: torch.device, stream: int) -> None:
    with _LOCK:
        # smaller sets of the stream that nobody holds have no use beside this one
        _FREE[:] = [f for f in _FREE if f[:2] != (device.index, stream) or f[2][1].numel() >= ws[1].numel()][1 - _KEEP:]
        _FREE.append((device.index, stream, ws))


def _as(t: torch.Tensor, dtype: torch.dtype) -> torch.Tensor:
    return t if t.dtype == dtype and t.is_contiguous() else t.to(dtype).contiguous()


def filtered_topk(corpus: torch.Tensor, user_codes: torch.Tensor, dates: torch.Tensor, queries: torch.Tensor,
                  q_user: torch.Tensor, q_floor: torch.Tensor, ks: torch.Tensor, kmax: int,
                  cap: int = 65536) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """-> (row ids [nq,kmax] int32, scores [nq,kmax] f32, counts [nq] int32), best first."""
    nq, D = queries.shape
    if not N.use_native(corpus):
        return filtered_topk_ref(corpus, user_codes, dates, queries, q_user.tolist(), q_floor.tolist(),
                                 ks.tolist(), kmax)
    if nq > 64:  # kernel handles 64 queries per launch
        parts = [filtered_topk(corpus, user_codes, dates, queries[i:i + 64], q_user[i:i + 64], q_floor[i:i + 64],
                               ks[i:i + 64], kmax, cap) for i in range(0, nq, 64)]
        return tuple(torch.cat(x) for x in zip(*parts))
    cap = max(SORT_CAP, min(cap, corpus.shape[0]))
    stream = N.stream()
    ws = _take(nq * cap, corpus.device, stream)
    counts, cand, scores, oc = ws                                    # the lists: nq rows of cap entries; oc is written by the kernel itself
    # converted inputs bound to names: as N.ptr(x.to(...)) temporaries they would be freed before
    # the launch and the next conversion could reuse (overwrite) their memory on the stream
    qu, qf = _as(q_user, torch.int32), _as(q_floor, torch.int64)
    dev, cp = corpus.device, counts.data_ptr()
    N.call("penny_topk_filter", user_codes.data_ptr(), dates.data_ptr(), corpus.shape[0], D, qu.data_ptr(), qf.data_ptr(), nq, cp,
           cand.data_ptr(), cap, stream)
    # beside the filter: the results' memory
    queries, kk = _as(queries, torch.bfloat16), _as(ks, torch.int32)
    out_ids = torch.empty((nq, kmax), dtype=torch.int32, device=dev)
    out_scores = torch.empty((nq, kmax), dtype=torch.float32, device=dev)
    out_count = torch.empty((nq,), dtype=torch.int32, device=dev)
    N.call("penny_topk_rank", corpus.data_ptr(), D, queries.data_ptr(), kk.data_ptr(), nq, kmax, cp, cand.data_ptr(), scores.data_ptr(),
           cap, out_ids.data_ptr(), out_scores.data_ptr(), out_count.data_ptr(), oc.data_ptr(), stream)
    for i, c in enumerate(oc[:nq].tolist()):  # the call has waited for them; > SORT_CAP candidates: finish on device with torch.topk
        if c >= 0:
            continue
        total = -c
        k = min(int(ks[i]), total, kmax)
        if total <= cap:
            s, j = torch.topk(scores[i * cap:i * cap + total], k)
            out_ids[i, :k], out_scores[i, :k] = cand[i * cap:i * cap + total][j], s
        else:
            mask = (user_codes == q_user[i]) & (dates >= q_floor[i])
            full = (corpus.float() @ queries[i].float()).masked_fill(~mask, float("-inf"))
            s, j = torch.topk(full, k)
            out_ids[i, :k], out_scores[i, :k] = j.to(torch.int32), s
        out_count[i] = k
    _hand_back(ws, corpus.device, stream)
    return out_ids, out_scores, out_count
