"""Sequence-mixer ops of the hybrid decoders (``csrc/mixers``): a 32-bit residual stream with a fused
parallel-block update + RMS norm, grouped / gated RMS norms, the Mamba-2 causal convolution and
state-space scan over a flat batch of segments, latent attention over a paged latent cache with a
sliding window, clamped gated units, and biased top-k routing; and, for the sequential post-norm
decoders, a hashed token-pair embedding, layer norm on the sublayer output fused with the residual
add, matrix-state linear recurrences (gated linear attention, gated delta rule), a real-gated linear
recurrent unit, sliding-window attention with grouped key/value heads over a paged [k | v] row cache,
gated activations with a per-row scale and sigmoid top-k routing; and, for decoders with several
residual streams per token (hyper-connections), the fused stream update + read + RMS norm, a rotation
of projected heads (two pair layouts, scaled frequencies, per-head RMS norm), matrix-state recurrences
with one fixed decay per head, a chunked attention mask, top-k routing with a softmax over the chosen
logits, and the logit scale / soft cap; and, for pre-norm decoders with gated residual updates, a sigmoid
gate and two weighted outputs on the fused residual update, attention with kept first tokens beyond a
sliding window and with unnormalised sigmoid weights, a minimal gated recurrent unit, values blended
across layers at the cache write, and linearly scaled rotation frequencies; and, for decoders whose norms are
elementwise (dynamic tanh) on both sides of a sublayer, one pass that norms a sublayer's output into the
stream and the stream into the next sublayer's input, a short convolution fused with per-head norms, a query
temperature and the cache write, distance biases, softmax sinks and elementwise output gates in the attention,
and routing with renormalised, scaled weights; and, for decoders that run a span of layers several times, the
embedding output added again inside the residual update, a distance bias read from a table of logarithmic buckets,
soft-capped attention scores, whole-projection norms fused with a rotation, sinks in latent attention, and
frequencies scaled by their wavelength.

Activations are bf16 or f32 (a model-wide choice); statistics, scores, softmax, recurrences and the
residual stream are f32 either way.  CUDA(HIP) tensors run the kernels of ``libpenny_mixers.so``
and fail loudly without it; CPU tensors run the fp32 PyTorch forms below (CI).

Batch layout: a step's rows are ``S`` segments, segment ``s`` owning rows ``cu[s]:cu[s+1]`` (a
prompt chunk, or a single decoded token), ``pos`` the position of every row, ``slot[s]`` the
segment's recurrent-state slot (< 0: padding, skipped) and ``bt[s]`` its cache page table.  A
segment whose first row is at position 0 starts from zero state whatever its slot holds.
"""
from __future__ import annotations

import ctypes
import functools
from typing import NamedTuple, Optional, Tuple, Union

import torch
import torch.nn.functional as F

from . import _native as N
from .gemm import Slabs, project

PAGE = 64


def _dt(t: torch.Tensor) -> int:
    if t.dtype == torch.float32:
        return 1
    if t.dtype == torch.bfloat16:
        return 0
    raise TypeError(f"mixer ops take bf16 or f32 tensors, got {t.dtype}")


def _rows(t: torch.Tensor) -> torch.Tensor:
    """A 2-D view whose last dimension is contiguous (column slices of a projection pass as is)."""
    if t.dim() != 2 or t.stride(1) != 1:
        raise ValueError("expected a [rows, n] tensor with unit column stride")
    return t


# ----------------------------------------------------------------------------------------------
# residual stream
# ----------------------------------------------------------------------------------------------
class Routed(NamedTuple):
    """A routed feed-forward's output whose rows the norm behind it adds up (the operands of :func:`moe_combine`)."""
    ys: torch.Tensor
    pos: torch.Tensor
    idx: torch.Tensor
    wts: Optional[torch.Tensor]
    h: torch.Tensor
    shared: Union[torch.Tensor, Slabs, None]
    num_experts: int
    identity: bool = True        # entries >= num_experts may occur

    @property
    def dtype(self) -> torch.dtype:
        return self.ys.dtype

    def materialize(self) -> torch.Tensor:
        return moe_combine(self.ys, self.pos, self.idx, self.wts, self.h, whole(self.shared), self.num_experts)


Sublayer = Union[torch.Tensor, Slabs, Routed]


def whole(v: Optional[Sublayer]) -> Optional[torch.Tensor]:
    """A sublayer's output written out."""
    return v if v is None or isinstance(v, torch.Tensor) else v.materialize()


class _Part(ctypes.Structure):
    """``MxPart`` of ``csrc/mixers/mx_common.h``."""
    _fields_ = [("p", ctypes.c_void_p), ("ld", ctypes.c_long), ("slab", ctypes.c_long), ("ys", ctypes.c_void_p), ("sy", ctypes.c_long),
                ("pos", ctypes.c_void_p), ("idx", ctypes.c_void_p), ("wts", ctypes.c_void_p), ("h", ctypes.c_void_p), ("sh", ctypes.c_long),
                ("slabs", ctypes.c_int), ("E", ctypes.c_int), ("top", ctypes.c_int)]


def _by_four(t: torch.Tensor) -> bool:
    ld, one = t.stride()
    return one == 1 and ld % 4 == 0 and t.data_ptr() % (16 if t.dtype == torch.float32 else 8) == 0


def _part(v: Sublayer, T: int, W: int) -> Optional[_Part]:
    """The parts of a sublayer output [T, W] for the kernels that add them up, or None: rows that they do not read by four."""
    r = v if isinstance(v, Routed) else None
    base = v if r is None else r.shared
    p, ld, slab, slabs = None, 0, 0, 0
    if base is not None:
        if base.shape != (T, W) or base.dtype != v.dtype:
            raise ValueError(f"a sublayer's output is [{T}, {W}], all of one type")
        if isinstance(base, Slabs):
            p, ld, slab, slabs = base.P.data_ptr(), W, T * W, base.P.shape[0]
            if p % 16 or not base.P.is_contiguous():
                return None
        elif _by_four(base):
            p, ld = base.data_ptr(), base.stride(0)
        else:
            return None
    if r is None:
        return _Part(p, ld, slab, None, 0, None, None, None, None, 0, slabs, 0, 0)
    ys, pos, idx, wts, h = r[:5]
    many = idx.shape
    if len(many) != 2 or many[0] != T or pos.shape != many or ys.shape[1] != W or h.shape != (T, W) or ys.dtype != h.dtype or \
            (wts is not None and wts.shape != many):
        raise ValueError("a routed output has an entry per token and choice")
    if not (_by_four(ys) and _by_four(h) and idx.is_contiguous() and pos.is_contiguous() and (wts is None or wts.is_contiguous())):
        return None
    # (no identity entries: h, which may be the stream that is written, is not read)
    return _Part(p, ld, slab, ys.data_ptr(), ys.stride(0), pos.data_ptr(), idx.data_ptr(), N.ptr(wts), h.data_ptr() if r.identity else None,
                 h.stride(0), slabs, r.num_experts if r.identity else 0x7fffffff, many[1])


def _parts(x: torch.Tensor, a: Optional[Sublayer], b: Optional[Sublayer], widest: int):
    """(parts of a, parts of b) where a kernel of rows up to ``widest`` columns adds them up into ``x``, else None."""
    if (a is None or type(a) is torch.Tensor) and (b is None or type(b) is torch.Tensor):
        return None
    T, W = x.shape
    if a is None or W % 4 or W > widest or x.data_ptr() % 16 or (b is not None and a.dtype != b.dtype) or not N.use_native(x):
        return None
    for v in (a, b):
        if isinstance(v, Routed) and v.identity and v.h.untyped_storage().data_ptr() == x.untyped_storage().data_ptr():
            return None
    p = _part(a, T, W)
    if p is None or b is None:
        return None if p is None else (ctypes.byref(p), None)
    q = _part(b, T, W)
    return None if q is None else (ctypes.byref(p), ctypes.byref(q))


def embed_f32(ids: torch.Tensor, table: torch.Tensor) -> torch.Tensor:
    """Token rows of ``table`` (bf16 or f32) as an f32 residual stream [T, W]."""
    T, (V, W) = ids.numel(), table.shape
    if N.use_native(table):
        out = torch.empty((T, W), dtype=torch.float32, device=table.device)
        N.mcall("mx_embed", N.ptr(ids.to(torch.int32).contiguous()), N.ptr(table), _dt(table), N.ptr(out), T, W, V,
                N.stream())
        return out
    return table[ids.long().clamp(0, V - 1)].float()


def residual_norm(x: torch.Tensor, w: Optional[torch.Tensor], eps: float, a: Optional[Sublayer] = None,
                  b: Optional[Sublayer] = None, mult: float = 1.0,
                  out_dtype: torch.dtype = torch.bfloat16, mult_b: Optional[float] = None,
                  gate: Optional[torch.Tensor] = None, gate_bias: Optional[torch.Tensor] = None,
                  ids: Optional[torch.Tensor] = None, table: Optional[torch.Tensor] = None) -> Optional[torch.Tensor]:
    """``x`` (f32 [T, W], in place) <- x + mult * (a + b) when a sublayer output is given, then
    y = x / sqrt(mean(x^2) + eps) * w in ``out_dtype`` (``w`` None: the update only).  ``mult_b``: b's own
    weight, the update is mult * a + mult_b * b.  ``gate`` ([T, W] column slice, the type of a) and
    ``gate_bias`` (f32 [W]): the update is multiplied element by element by sigmoid(gate + gate_bias).
    ``ids`` (int32 [T]) with ``table`` ([vocab, W], the type of a): the row ``table[ids]`` is added after the update."""
    return _residual_norm(x, w, eps, a, b, mult, out_dtype, mult_b, gate, gate_bias, ids, table, False)


def embed_norm(ids: torch.Tensor, table: torch.Tensor, w: torch.Tensor, eps: float,
               out_dtype: torch.dtype = torch.bfloat16) -> Tuple[torch.Tensor, torch.Tensor]:
    """Token rows of ``table`` as an f32 residual stream x [T, W] and its RMS norm in ``out_dtype``, in one pass."""
    x = torch.empty((ids.numel(), table.shape[1]), dtype=torch.float32, device=table.device)
    h = _residual_norm(x, w, eps, None, None, 1.0, out_dtype, None, None, None, ids, table, True)
    return x, h


def _residual_norm(x, w, eps, a, b, mult, out_dtype, mult_b, gate, gate_bias, ids, table, fresh):
    T, W = x.shape
    assert x.dtype == torch.float32 and x.is_contiguous()
    mult_b = mult if mult_b is None else mult_b
    parts = _parts(x, a, b, 8192) if gate is None and table is None and w is not None and w.data_ptr() % 16 == 0 else None
    if parts is not None:
        out = torch.empty((T, W), dtype=out_dtype, device=x.device)
        N.mcall("mx_residual_norm_parts", N.ptr(x), parts[0], parts[1], int(a.dtype == torch.float32), float(mult), float(mult_b), N.ptr(w),
                float(eps), N.ptr(out), _dt(out), T, W, N.stream())
        return out
    a, b = whole(a), whole(b)
    ab = a if a is not None else b
    if gate is not None and ab is None:
        raise ValueError("a gate needs a sublayer output to act on")
    if table is not None and (ids is None or ids.numel() != T or table.shape[1] != W):
        raise ValueError("table: one id per row and rows of the stream's width")
    if N.use_native(x):
        out = torch.empty((T, W), dtype=out_dtype, device=x.device) if w is not None else None
        if a is not None and b is not None:
            assert a.dtype == b.dtype
        if gate is not None:
            assert gate.dtype == ab.dtype and gate.shape[1] == W
        if table is not None:
            assert table.is_contiguous() and (ab is None or table.dtype == ab.dtype)
            ids = ids.to(torch.int32).contiguous()
        src = ab if ab is not None else table
        N.mcall("mx_residual_norm", N.ptr(x), N.ptr(_rows(a)) if a is not None else None,
                a.stride(0) if a is not None else 0, N.ptr(_rows(b)) if b is not None else None,
                b.stride(0) if b is not None else 0, _dt(src) if src is not None else 1, float(mult), float(mult_b),
                N.ptr(_rows(gate)) if gate is not None else None, gate.stride(0) if gate is not None else 0,
                N.ptr(gate_bias), N.ptr(ids) if table is not None else None, N.ptr(table),
                table.shape[0] if table is not None else 0, 1 if fresh else 0, N.ptr(w), float(eps), N.ptr(out), _dt(out) if out is not None else 1, T, W, N.stream())
        return out
    if ab is not None:
        s = torch.zeros_like(x)
        for t, m in ((a, mult), (b, mult_b)):
            if t is not None:
                s = s + m * t.float()
        if gate is not None:
            s = s * torch.sigmoid(gate.float() + (gate_bias.float() if gate_bias is not None else 0.0))
        x.add_(s)
    if table is not None:
        row = table[ids.long().clamp(0, table.shape[0] - 1)].float()
        if fresh:
            x.copy_(row)
        else:
            x.add_(row)
    if w is None:
        return None
    return (x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * w.float()).to(out_dtype)


class DynTanh(NamedTuple):
    """Parameters of the elementwise norm tanh(alpha * x) * w + b (no statistics): ``w`` and ``b`` f32 [W]."""
    alpha: float
    w: torch.Tensor
    b: torch.Tensor

    def plain(self, v: torch.Tensor) -> torch.Tensor:
        return torch.tanh(self.alpha * v) * self.w.float() + self.b.float()


def _dyn_tanh_call(x, a, ids, table, scale, pre, post, out):
    T, W = x.shape
    src = a if a is not None else table
    N.mcall("mx_dyn_tanh", N.ptr(x), N.ptr(_rows(a)) if a is not None else None, a.stride(0) if a is not None else 0,
            N.ptr(ids), N.ptr(table), table.shape[0] if table is not None else 0, float(scale),
            _dt(src) if src is not None else 1, pre.alpha if pre is not None else 0.0, N.ptr(pre.w) if pre is not None else None,
            N.ptr(pre.b) if pre is not None else None, post.alpha if post is not None else 0.0,
            N.ptr(post.w) if post is not None else None, N.ptr(post.b) if post is not None else None, N.ptr(out),
            _dt(out) if out is not None else 1, T, W, N.stream())


def dyn_tanh_embed(ids: torch.Tensor, table: torch.Tensor, scale: float, norm: DynTanh, post: Optional[DynTanh] = None,
                   out_dtype: torch.dtype = torch.bfloat16) -> Tuple[torch.Tensor, Optional[torch.Tensor]]:
    """The f32 residual stream x = norm(table[id] * scale) [T, W] and, with ``post``, post(x) in ``out_dtype`` (the
    first sublayer's input), in one pass."""
    T, (V, W) = ids.numel(), table.shape
    if N.use_native(table):
        x = torch.empty((T, W), dtype=torch.float32, device=table.device)
        out = torch.empty((T, W), dtype=out_dtype, device=table.device) if post is not None else None
        _dyn_tanh_call(x, None, ids.to(torch.int32).contiguous(), table.contiguous(), scale, norm, post, out)
        return x, out
    x = norm.plain(table[ids.long().clamp(0, V - 1)].float() * scale)
    return x, post.plain(x).to(out_dtype) if post is not None else None


def dyn_tanh_residual(x: torch.Tensor, y: Optional[Sublayer], norm: Optional[DynTanh], post: Optional[DynTanh] = None,
                      out_dtype: torch.dtype = torch.bfloat16) -> Optional[torch.Tensor]:
    """``x`` (f32 [T, W], in place) <- x + norm(y) for a sublayer's output ``y`` (None: x stays), then post(x) in
    ``out_dtype`` (the next sublayer's input; ``post`` None: the update only), in one pass."""
    T, W = x.shape
    parts = _parts(x, y, None, 1 << 30) if norm is not None and all(
        (d.w.data_ptr() | d.b.data_ptr()) % 16 == 0 for d in (norm, post) if d is not None) else None
    if parts is not None:
        assert x.dtype == torch.float32 and x.is_contiguous()
        out = torch.empty((T, W), dtype=out_dtype, device=x.device) if post is not None else None
        N.mcall("mx_dyn_tanh_parts", N.ptr(x), parts[0], int(y.dtype == torch.float32), norm.alpha, N.ptr(norm.w), N.ptr(norm.b),
                post.alpha if post is not None else 0.0, N.ptr(post.w) if post is not None else None,
                N.ptr(post.b) if post is not None else None, N.ptr(out), _dt(out) if out is not None else 1, T, W, N.stream())
        return out
    y = whole(y)
    assert x.dtype == torch.float32 and x.is_contiguous() and (y is None or (y.shape == x.shape and norm is not None))
    if N.use_native(x):
        out = torch.empty((T, W), dtype=out_dtype, device=x.device) if post is not None else None
        _dyn_tanh_call(x, y, None, None, 1.0, norm if y is not None else None, post, out)
        return out
    if y is not None:
        x.add_(norm.plain(y.float()))
    return post.plain(x).to(out_dtype) if post is not None else None


def group_norm(inp: torch.Tensor, w: torch.Tensor, eps: float, groups: int = 1, gate: Optional[torch.Tensor] = None,
               out_dtype: Optional[torch.dtype] = None) -> torch.Tensor:
    """RMS norm of each of ``groups`` equal parts of every row of ``inp`` [T, n] (each part by its own
    root mean square), times ``w`` [n].  ``gate``: the row is multiplied by silu(gate) first."""
    T, n = inp.shape
    out_dtype = out_dtype or inp.dtype
    if n % groups:
        raise ValueError(f"{n} columns do not split into {groups} groups")
    if N.use_native(inp):
        out = torch.empty((T, n), dtype=out_dtype, device=inp.device)
        N.mcall("mx_group_norm", N.ptr(_rows(inp)), inp.stride(0), _dt(inp), N.ptr(_rows(gate)) if gate is not None else None,
                gate.stride(0) if gate is not None else 0, _dt(gate) if gate is not None else 1, N.ptr(w),
                float(eps), N.ptr(out), out.stride(0), _dt(out), T, groups, n // groups, N.stream())
        return out
    v = inp.float()
    if gate is not None:
        v = v * F.silu(gate.float())
    v = v.view(T, groups, n // groups)
    v = v * torch.rsqrt(v.pow(2).mean(-1, keepdim=True) + eps)
    return (v.reshape(T, n) * w.float()).to(out_dtype)


# ----------------------------------------------------------------------------------------------
# activations
# ----------------------------------------------------------------------------------------------
def relu2(x: torch.Tensor) -> torch.Tensor:
    """relu(x)^2, rows may be a column slice of a wider projection."""
    T, n = x.shape
    if N.use_native(x):
        out = torch.empty((T, n), dtype=x.dtype, device=x.device)
        N.mcall("mx_relu2", N.ptr(_rows(x)), x.stride(0), N.ptr(out), out.stride(0), _dt(x), T, n, N.stream())
        return out
    return torch.relu(x.float()).square().to(x.dtype)


def glu_clamp(gate: torch.Tensor, up: torch.Tensor, limit: float, alpha: float) -> torch.Tensor:
    """g = min(gate, limit), u = clamp(up, -limit, limit): g * sigmoid(alpha * g) * (u + 1)."""
    T, n = gate.shape
    if N.use_native(gate):
        out = torch.empty((T, n), dtype=gate.dtype, device=gate.device)
        N.mcall("mx_glu_clamp", N.ptr(_rows(gate)), gate.stride(0), N.ptr(_rows(up)), up.stride(0), float(limit),
                float(alpha), N.ptr(out), out.stride(0), _dt(gate), T, n, N.stream())
        return out
    g = gate.float().clamp(max=limit)
    u = up.float().clamp(-limit, limit)
    return (g * torch.sigmoid(alpha * g) * (u + 1)).to(gate.dtype)


# ----------------------------------------------------------------------------------------------
# routing
# ----------------------------------------------------------------------------------------------
def route_biased(z: torch.Tensor, bias: Optional[torch.Tensor], top: int, score: str = "softmax", renorm: bool = False,
                 scale: float = 1.0) -> Tuple[torch.Tensor, torch.Tensor]:
    """Scores s of the f32 router logits ``z``: softmax over all entries, or (``score="sigmoid"``) the sigmoid of
    each; the ``top`` entries with the largest s + bias are chosen, and their weights are the unbiased scores s --
    with ``renorm`` divided by the chosen scores' sum (+ 1e-20) -- times ``scale``.  Returns (weights f32
    [T, top], indices int32 [T, top])."""
    T, E = z.shape
    assert z.dtype == torch.float32
    if score not in ("softmax", "sigmoid"):
        raise ValueError(f"unknown routing score {score!r}")
    if N.use_native(z):
        z = z.contiguous()
        w = torch.empty((T, top), dtype=torch.float32, device=z.device)
        i = torch.empty((T, top), dtype=torch.int32, device=z.device)
        N.mcall("mx_route_biased", N.ptr(z), N.ptr(bias), E, top, 1 if score == "sigmoid" else 0, 1 if renorm else 0,
                float(scale), N.ptr(w), N.ptr(i), T, N.stream())
        return w, i
    s = torch.sigmoid(z) if score == "sigmoid" else torch.softmax(z, -1)
    c = s + bias.float() if bias is not None else s
    # a stable sort: ties go to the lower index, as in the kernel
    idx = torch.sort(c, dim=-1, descending=True, stable=True).indices[:, :top]
    w = s.gather(1, idx)
    if renorm:
        w = w / (w.sum(-1, keepdim=True) + 1e-20)
    return w * scale, idx.to(torch.int32)


def router_takes(T: int, E: int, W: int, f32: bool) -> bool:
    """Is ``mx_router`` the faster way for ``T`` rows, ``E`` entries, ``W`` columns?  Its kernels work in sixteens of entries (figures beside
    them): up to 32 entries always; up to 48 in matrices that it reads faster than the library's three launches start; beyond, by one row
    per block or on the matrix cores and in yet narrower ones.  f32 has no conversion to save and no matrix form."""
    if W % 32 or W > 8192 or E > 64 or (f32 and T > 1024):
        return False
    if E <= 32:
        return True
    if E <= 48:
        return W <= 2048 or (W <= 4096 and T <= (256 if f32 else 1024))
    if T <= 256:
        return W <= (1024 if f32 else 2048)
    return T > 1024 and (W <= 1024 or (W <= 2048 and T <= 4096))


class Glu(NamedTuple):
    """Operands of :func:`glu_clamp` that a router's launch may take along."""
    gate: torch.Tensor
    up: torch.Tensor
    limit: float
    alpha: float


def _router(h: torch.Tensor, w: torch.Tensor, zbias, bias, biased: bool, top: int, score: str, renorm: bool, scale: float, glu: Optional[Glu] = None):
    """(weights, indices, act) by ``mx_router`` where it serves the call (up to 64 entries, whole groups of 32 columns, 16-byte rows) and is the
    faster way (:func:`router_takes`), else None.  act: :func:`glu_clamp` of ``glu`` where its rows are in whole 16 bytes, else None."""
    T, W = h.shape
    E = w.shape[0]
    es = h.element_size()
    if not N.use_native(h) or T == 0 or h.dtype not in (torch.bfloat16, torch.float32) or not router_takes(T, E, W, h.dtype == torch.float32) or \
            not w.is_contiguous() or h.stride(1) != 1 or h.stride(0) * es % 16 or h.data_ptr() % 16 or w.data_ptr() % 16:
        return None
    outw = torch.empty((T, top), dtype=torch.float32, device=h.device)
    outi = torch.empty((T, top), dtype=torch.int32, device=h.device)
    act, more = None, (None, 0, None, 0, 0.0, 0.0, None, 0)
    if glu is not None:
        g, u = glu.gate, glu.up
        n, (sg, one), (su, one_) = g.shape[1], g.stride(), u.stride()
        if g.shape == u.shape and g.shape[0] == T and g.dtype == u.dtype == h.dtype and one == one_ == 1 and n > 0 and \
                (n * es | sg * es | su * es | g.data_ptr() | u.data_ptr()) % 16 == 0 and T * n < 1 << 36:
            act = torch.empty((T, n), dtype=h.dtype, device=h.device)
            more = (g.data_ptr(), sg, u.data_ptr(), su, float(glu.limit), float(glu.alpha), act.data_ptr(), n)
    N.mcall("mx_router", N.ptr(h), h.stride(0), _dt(h), N.ptr(w), N.ptr(zbias), N.ptr(bias), 1 if biased else 0, ROUTE_SCORES[score],
            1 if renorm else 0, float(scale), E, top, W, N.ptr(outw), N.ptr(outi), *more, T, N.stream())
    return outw, outi, act


def router_biased(h: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor], top: int, score: str = "softmax",
                  renorm: bool = False, scale: float = 1.0) -> Tuple[torch.Tensor, torch.Tensor]:
    """:func:`route_biased` of the logits ``h w^T`` in f32 (``h`` [T, W] bf16 or f32, ``w`` f32 [E, W])."""
    return router_glu(h, w, bias, top, score, renorm, scale)[:2]


def router_scores(h: torch.Tensor, w: torch.Tensor, zbias: Optional[torch.Tensor], top: int,
                  score: str = "sigmoid") -> Tuple[torch.Tensor, torch.Tensor]:
    """:func:`route_scores` of the logits ``h w^T + zbias`` in f32."""
    assert w.dtype == torch.float32 and w.shape[1] == h.shape[1] and 1 <= top <= w.shape[0]
    if score not in ROUTE_SCORES:
        raise ValueError(f"unknown routing score {score!r}")
    r = _router(h, w, zbias, None, False, top, score, False, 1.0)
    return r[:2] if r is not None else route_scores(F.linear(h.float(), w, zbias), top, score)


def router_glu(h: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor], top: int, score: str = "softmax", renorm: bool = False,
               scale: float = 1.0, glu: Optional[Glu] = None) -> Tuple[torch.Tensor, torch.Tensor, Optional[torch.Tensor]]:
    """:func:`router_biased` and, given, :func:`glu_clamp` of ``glu``, in one launch where one serves both."""
    assert w.dtype == torch.float32 and w.shape[1] == h.shape[1] and 1 <= top <= w.shape[0]
    if score not in ("softmax", "sigmoid"):
        raise ValueError(f"unknown routing score {score!r}")
    r = _router(h, w, None, bias, True, top, score, renorm, scale, glu)
    if r is None:
        r = *route_biased(F.linear(h.float(), w), bias, top, score, renorm, scale), None
    return r if glu is None or r[2] is not None else (r[0], r[1], glu_clamp(*glu))


class ExpertRows(NamedTuple):
    """The matrices of all experts as :func:`experts` reads them (see :func:`pack_experts`)."""
    data: torch.Tensor      # [experts, row groups, K steps of 64 bytes, 4, 16, elements per 16 bytes]
    rows: int               # rows of one matrix
    parts: int              # 2: gate and up in turns of 16 rows


def pack_experts(mats, dtype: torch.dtype) -> ExpertRows:
    """``mats``: per expert one matrix [out, in], or the pair (gate, up).  Rows in groups of 16 (a pair's groups take
    turns) and K in pieces of 64 bytes, each piece stored as the matrix instruction's lanes read it; rows and K are
    padded with zeros to whole groups and 128 bytes."""
    pairs = [m if isinstance(m, (tuple, list)) else (m,) for m in mats]
    E, parts, (n, k) = len(pairs), len(pairs[0]), pairs[0][0].shape
    el = 16 // torch.empty((), dtype=dtype).element_size()
    groups, kp = -(-n // 16), -(-k // (8 * el)) * 8 * el
    full = torch.stack([m.to(dtype) for ms in pairs for m in ms])
    if (groups * 16, kp) != (n, k):
        full = F.pad(full, (0, kp - k, 0, groups * 16 - n))
    data = full.view(E, parts, groups, 16, kp // (4 * el), 4, el).permute(0, 2, 1, 4, 5, 3, 6).contiguous()
    return ExpertRows(data.view(E, groups * parts, kp // (4 * el), 4, 16, el), n, parts)


EXPERT_UNITS = {"clamped": 1, "silu": 2, "gelu_tanh": 3, "relu2": 4}


def experts(h: torch.Tensor, idx: torch.Tensor, w1: ExpertRows, w2: ExpertRows, unit: str, limit: float = 0.0, alpha: float = 0.0,
            scale: Optional[torch.Tensor] = None) -> Tuple[torch.Tensor, torch.Tensor]:
    """Every token's chosen experts (GPU only): rows ys[pos[t, k]] = W2_e unit(W1_e h[t]) for e = idx[t, k] < experts
    (identity experts have no row).  ``unit``: "clamped" (g, u of :func:`glu_clamp` with ``limit`` and ``alpha``),
    "silu" / "gelu_tanh" (act(s g) * (s u), s the pair's entry of ``scale`` f32 [T, top] or 1) or "relu2" (one
    matrix).  No host read: the rows are sorted by expert on the device.  Returns (ys, pos int32 [T, top])."""
    T, W = h.shape
    top, E = idx.shape[1], w1.data.shape[0]
    el = w1.data.shape[-1]
    assert h.dtype == w1.data.dtype == w2.data.dtype and idx.dtype == torch.int32 and idx.is_contiguous()
    assert scale is None or (scale.dtype == torch.float32 and scale.is_contiguous() and scale.shape == idx.shape)
    wp = -(-W // el) * el
    if wp != W:                                   # rows in whole 16-byte units
        h = F.pad(h, (0, wp - W))
    elif h.stride(1) != 1 or h.stride(0) % el or h.data_ptr() % 16:
        h = h.contiguous()
    P = T * top
    lda = -(-w1.rows // el) * el
    act = torch.empty((P, lda), dtype=h.dtype, device=h.device)
    ys = torch.empty((P, wp), dtype=h.dtype, device=h.device)
    # pos | sorted row -> pair | row tiles of (expert, first row, rows, -), at most P / 16 + experts of them
    ws = torch.empty(2 * (-(-P // 4) * 4) + 4 * (P // 16 + min(P, E) + 1), dtype=torch.int32, device=h.device)
    N.mcall("mx_experts", N.ptr(h), h.stride(0), N.ptr(idx), T, top, E, wp, w1.rows, N.ptr(w1.data), w1.data.shape[2],
            w1.data.shape[1], N.ptr(w2.data), w2.data.shape[2], w2.data.shape[1], EXPERT_UNITS[unit], float(limit),
            float(alpha), N.ptr(scale), N.ptr(act), lda, N.ptr(ys), N.ptr(ws), _dt(h), N.stream())
    return ys[:, :W], ws[:P].view(T, top)


def moe_combine(ys: Optional[torch.Tensor], pos: torch.Tensor, idx: torch.Tensor, wts: Optional[torch.Tensor], h: torch.Tensor,
                shared: Optional[torch.Tensor], num_experts: int) -> torch.Tensor:
    """out[t] = sum_k wts[t, k] * src(t, k) (+ shared[t]): src is the token's own input ``h[t]`` for an
    identity expert (idx >= num_experts), else row ``pos[t, k]`` of the expert outputs ``ys``; ``wts`` None: ones."""
    T, W = h.shape
    top = idx.shape[1]
    if N.use_native(h):
        out = torch.empty((T, W), dtype=h.dtype, device=h.device)
        pos, idx, wts = pos.contiguous(), idx.contiguous(), wts.contiguous() if wts is not None else None
        N.mcall("mx_moe_combine", N.ptr(_rows(ys)) if ys is not None else None, ys.stride(0) if ys is not None else 0,
                N.ptr(pos), N.ptr(idx), N.ptr(wts),
                N.ptr(_rows(h)), h.stride(0), N.ptr(_rows(shared)) if shared is not None else None,
                shared.stride(0) if shared is not None else 0, num_experts, top, W, N.ptr(out), _dt(h), T, N.stream())
        return out
    acc = shared.float().clone() if shared is not None else torch.zeros((T, W), dtype=torch.float32)
    for k in range(top):
        e = idx[:, k].long()
        ident = e >= num_experts
        src = h.float().clone()
        if ys is not None and (~ident).any():
            rows = pos[:, k].long().clamp(0, ys.shape[0] - 1)
            src = torch.where(ident[:, None], src, ys.float()[rows])
        acc += (wts[:, k:k + 1] if wts is not None else 1.0) * src
    return acc.to(h.dtype)


# ----------------------------------------------------------------------------------------------
# state-space mixer
# ----------------------------------------------------------------------------------------------
def conv_silu(inp: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor], state: torch.Tensor,
              cu: torch.Tensor, slot: torch.Tensor, pos: torch.Tensor, max_len: int) -> torch.Tensor:
    """Causal per-channel convolution + SiLU over every segment.  ``inp`` [T, C] (a column slice of the
    in-projection), ``w`` f32 [C, K] (last column: the current token's tap), ``state`` f32
    [slots, K-1, C]: the last K-1 inputs of each slot's sequence, read (unless the segment starts
    at position 0) and then replaced.  Returns f32 [T, C]."""
    T, C = inp.shape
    K = w.shape[1]
    S = cu.numel() - 1
    if N.use_native(inp):
        out = torch.empty((T, C), dtype=torch.float32, device=inp.device)
        N.mcall("mx_conv_silu", N.ptr(_rows(inp)), inp.stride(0), _dt(inp), N.ptr(w), N.ptr(bias), N.ptr(state),
                N.ptr(cu), N.ptr(slot), N.ptr(pos), N.ptr(out), S, int(max_len), T, C, K, N.stream())
        return out
    out = torch.zeros((T, C), dtype=torch.float32)
    cul, sll, pl = cu.tolist(), slot.tolist(), pos.tolist()
    x = inp.float()
    for s in range(S):
        a, b = cul[s], cul[s + 1]
        if sll[s] < 0 or b <= a:
            continue
        hist = torch.zeros((K - 1, C)) if pl[a] == 0 else state[sll[s]].clone()
        full = torch.cat([hist, x[a:b]])
        win = full.unfold(0, K, 1)                      # [n, C, K]
        acc = (win * w.float()[None]).sum(-1)
        if bias is not None:
            acc = acc + bias.float()
        out[a:b] = F.silu(acc)
        if K > 1:
            state[sll[s]] = full[-(K - 1):]
    return out


def _ssm_in_chunks(T: int, S: int, max_len: int, state: int) -> bool:
    """Whether a step of S segments and T rows goes in chunks rather than token by token (``state``: numbers in a state).

    An estimate of both forms' times in us.  Token by token: the longest chain, or the rows (staged by 32) and the states
    moved, about added where they are alike.  In chunks: three launches more, the products (64 rows at a time) and the same
    states, moved by single rows after the chunks and not beside them.  64 heads of 64 x 128, tokens / chunks: one segment of
    48 rows 17.9 / 17.6, of 64 20.7 / 18.1, of 256 69 / 28; four of 32 27.5 / 29.8, of 40 38 / 32; one of 64 beside 8 single
    rows 24 / 27, of 96 32 / 30; one of 192 beside 64 single rows 76 / 81, of 256 90 / 84.  32 heads: one of 64 beside 8
    single rows 21 / 24; four of 96 beside 64 55 / 61, of 128 64 / 61."""
    if max_len < 32:
        return False
    size = state / (64 * 64 * 128)
    moved = 0.75 * S * size
    staged, padded = (-(-max_len // n) * n / max_len for n in (32, 64))
    tokens = ((5.5 + 0.27 * max_len) ** 4 + (0.165 * max(T - S, 0) * staged * size + moved) ** 4) ** 0.25
    return 16.5 + 0.2 * S + 0.047 * T * padded * size + moved < tokens


def ssm_scan(u: torch.Tensor, dt_raw: torch.Tensor, dt_bias: torch.Tensor, A_log: torch.Tensor, D: torch.Tensor,
             state: torch.Tensor, cu: torch.Tensor, slot: torch.Tensor, pos: torch.Tensor, heads: int, vdim: int,
             nstate: int, groups: int, max_len: int = 0) -> torch.Tensor:
    """Mamba-2 recurrence in f32 (``max_len``: no segment is longer, all rows when left out; steps of long segments go in
    chunks).  ``u`` f32 [T, H*P + 2*G*N] = [x | B | C] (after the convolution), ``dt_raw`` [T, H]; per head h of group
    h // (H / G):
    dt = softplus(dt_raw + dt_bias), S <- exp(-exp(A_log) dt) S + dt x B^T, y = S C + D x.
    ``state`` f32 [slots, H, P, N] is read (unless the segment starts at position 0) and replaced."""
    T, C = u.shape
    H, P, Ns, G = heads, vdim, nstate, groups
    S = cu.numel() - 1
    assert u.dtype == torch.float32 and u.is_contiguous() and C == H * P + 2 * G * Ns
    if N.use_native(u):
        y = torch.empty((T, H * P), dtype=torch.float32, device=u.device)
        max_len = max_len or T
        ws = None
        if Ns in (64, 128, 256) and _ssm_in_chunks(T, S, max_len, H * P * Ns):          # the factors: ssd_chunk_floats of the kernels
            ws = torch.empty((max(1, T // 64 + min(S, T // 32)), G * 64 * (64 + 2 * Ns) + H * 2688), dtype=torch.float32, device=u.device)
        N.mcall("mx_ssm_scan", N.ptr(u), C, N.ptr(_rows(dt_raw)), dt_raw.stride(0), _dt(dt_raw), N.ptr(dt_bias),
                N.ptr(A_log), N.ptr(D), N.ptr(state), N.ptr(cu), N.ptr(slot), N.ptr(pos), N.ptr(y), S, int(max_len), H, P, Ns, G,
                T, N.ptr(ws), N.stream())
        return y
    y = torch.zeros((T, H * P), dtype=torch.float32)
    cul, sll, pl = cu.tolist(), slot.tolist(), pos.tolist()
    A = -torch.exp(A_log.float())
    rep = H // G
    for s in range(S):
        a, b = cul[s], cul[s + 1]
        if sll[s] < 0 or b <= a:
            continue
        St = torch.zeros((H, P, Ns)) if pl[a] == 0 else state[sll[s]].clone()
        dt = F.softplus(dt_raw[a:b].float() + dt_bias.float())          # [n, H]
        dec = torch.exp(A * dt)
        x = u[a:b, :H * P].view(-1, H, P)
        Bm = u[a:b, H * P:H * P + G * Ns].view(-1, G, Ns).repeat_interleave(rep, 1)
        Cm = u[a:b, H * P + G * Ns:].view(-1, G, Ns).repeat_interleave(rep, 1)
        for t in range(b - a):
            St = dec[t, :, None, None] * St + (dt[t, :, None] * x[t])[:, :, None] * Bm[t][:, None, :]
            y[a + t] = ((St * Cm[t][:, None, :]).sum(-1) + D.float()[:, None] * x[t]).reshape(-1)
        state[sll[s]] = St
    return y


# ----------------------------------------------------------------------------------------------
# latent attention
# ----------------------------------------------------------------------------------------------
def rope_inv_freq(dims: int, base: float, device=None) -> torch.Tensor:
    """f_i = base^(-2i / dims), i < dims / 2, f32."""
    i = torch.arange(0, dims, 2, dtype=torch.float32, device=device)
    return (1.0 / (base ** (i / dims))).contiguous()


def _rotate(v: torch.Tensor, ang: torch.Tensor, dims: int, m: float = 1.0) -> torch.Tensor:
    """Interleaved-pair rotation of the first ``dims`` entries of the last axis; ``ang`` broadcasts
    against v[..., 0:dims:2]."""
    out = v.clone()
    a, b = v[..., 0:dims:2], v[..., 1:dims:2]
    c, s = torch.cos(ang) * m, torch.sin(ang) * m
    out[..., 0:dims:2] = a * c - b * s
    out[..., 1:dims:2] = b * c + a * s
    return out


def latent_prep(kv: torch.Tensor, norm_w: torch.Tensor, eps: float, inv_freq: torch.Tensor, rot_dims: int,
                pos: torch.Tensor, slots: torch.Tensor, cache: torch.Tensor, q: torch.Tensor, heads: int,
                head_stride: int, rot_off: int, rank: int, rot_dim: int, mscale: float = 1.0) -> torch.Tensor:
    """Per token: c = RMSnorm(kv[:rank]) * norm_w and the rotated shared key part rope(kv[rank:]) go to
    cache row ``slots[t]`` (< 0: no write; ``cache`` [rows, rank + rot_dim]); every head's rotated
    query part ``q[t, h*head_stride + rot_off : +rot_dim]`` is rotated into the returned
    [T, heads, rot_dim].  Angles are pos * inv_freq in f32, pairs interleaved, cos and sin times ``mscale``."""
    T = kv.shape[0]
    R, Dr, H = rank, rot_dim, heads
    if N.use_native(kv):
        assert kv.dtype == cache.dtype == q.dtype
        q_rot = torch.empty((T, H, Dr), dtype=q.dtype, device=q.device)
        N.mcall("mx_latent_prep", N.ptr(_rows(kv)), kv.stride(0), N.ptr(norm_w), float(eps), N.ptr(inv_freq),
                int(rot_dims), float(mscale), N.ptr(pos), N.ptr(slots), N.ptr(cache), N.ptr(_rows(q)), q.stride(0), head_stride,
                rot_off, N.ptr(q_rot), _dt(kv), T, H, R, Dr, N.stream())
        return q_rot
    kvf = kv.float()
    c = kvf[:, :R]
    c = c * torch.rsqrt(c.pow(2).mean(-1, keepdim=True) + eps) * norm_w.float()
    ang = pos.float()[:, None] * inv_freq.float()[None, :rot_dims // 2]
    kr = _rotate(kvf[:, R:R + Dr], ang, rot_dims, mscale)
    rows = torch.cat([c, kr], 1).to(cache.dtype)
    ok = slots >= 0
    cache.view(-1, R + Dr)[slots[ok].long()] = rows[ok]
    qr = torch.stack([q[:, h * head_stride + rot_off:h * head_stride + rot_off + Dr] for h in range(H)], 1).float()
    return _rotate(qr, ang[:, None, :], rot_dims, mscale).to(q.dtype)


def _sink_softmax(sc: torch.Tensor, sink: Optional[torch.Tensor]) -> torch.Tensor:
    """Softmax over the last axis of f32 scores [n, H, keys]; ``sink`` [H]: one more entry of the denominator."""
    if sink is None:
        return torch.softmax(sc, -1)
    extra = sink.float()[None, :, None].expand(sc.shape[0], sc.shape[1], 1)
    return torch.softmax(torch.cat([sc, extra], -1), -1)[..., :-1]


class HeadLinear:
    """y[t, h] = W[h] x[t, h]: a matrix per head, ``w`` [H, N, K].  On the GPU the rows of heads are read and written where they lie
    (``mx_head_linear``); sizes that the kernel does not take (N in whole 16, rows of whole 64 bytes), those that it would serve
    slower (:meth:`_most_rows`) and the CPU go through a batched product."""

    def __init__(self, w: torch.Tensor):
        H, self.N, self.K = w.shape
        self.H, self.dtype = H, w.dtype
        self.native = N.use_native(w) and w.dtype in (torch.bfloat16, torch.float32) and self.N % 16 == 0 and \
            self.K * w.element_size() % 64 == 0 and H <= 65535
        self.most = self._most_rows()
        # the kernel's matrices, in whole 16 bytes, and the batched product's, whose right operand lies as it reads it: what calls need
        self.w = self.wt = None
        if self.most > 0:
            self.w = w.contiguous()
            if self.w.data_ptr() % 16:
                self.w = self.w.clone()
        if self.most < 1 << 40:
            self.wt = w.transpose(1, 2).contiguous()

    def _most_rows(self) -> int:
        """Rows that the kernel serves faster.  Every wave reads its columns of W for itself, so the library's tiles win where a head's
        matrix is large, or K is and the rows are many.  Us, batched product with its copies / here, heads x N x K: bf16 8 x 512 x 512 64
        rows 9.7 / 23.4, 8192 91 / 177; 16 x 256 x 256 64: 12.1 / 7.8, 8192: 82 / 97; 32 x 128 x 256 2048: 30 / 27, 8192: 105 / 98, 16384: 206 /
        223; 32 x 256 x 128 16384: 284 / 260; f32 16 x 96 x 256 2048: 28.5 / 27.0, 8192: 87 / 99; 32 x 128 x 256 512: 20.3 / 19.0, 2048: 56 / 60;
        16 x 256 x 96 16384: 276 / 218."""
        if not self.native or self.N * self.K > 32768:
            return 0
        return 1 << 40 if self.K <= self.N else (32768 if self.dtype == torch.float32 else 262144) // self.H

    def __call__(self, x: torch.Tensor) -> torch.Tensor:
        """x [T, H, K] (any strides) -> [T, H, N] contiguous."""
        T, H, K = x.shape
        if self.native and (x.dtype != self.dtype or (H, K) != (self.H, self.K)):
            raise ValueError("one row of the matrices' width per head, of their type")
        if T > self.most:
            return torch.bmm(x.transpose(0, 1), self.wt).transpose(0, 1).contiguous()
        es = x.element_size()
        if x.stride(2) != 1 or x.stride(0) * es % 16 or x.stride(1) * es % 16 or x.data_ptr() % 16:
            x = x.clone(memory_format=torch.contiguous_format)
        y = torch.empty((T, H, self.N), dtype=x.dtype, device=x.device)
        N.mcall("mx_head_linear", N.ptr(x), x.stride(0), x.stride(1), N.ptr(self.w), N.ptr(y), T, H, self.N, K, _dt(x), N.stream())
        return y

    def num_bytes(self) -> int:
        return sum(w.numel() * w.element_size() for w in (self.w, self.wt) if w is not None)


@functools.lru_cache(maxsize=1024)          # the estimate takes 1 - 5 us
def _key_parts(keys: int, blocks: int, most_blocks: int, pairs: int, width: int, dtype: torch.dtype) -> int:
    """How many blocks walk the keys of the same queries in the tiled attention (at most ``most_blocks`` over ``blocks``), for
    ``keys`` a query block may see and ``pairs`` (row, head) results of ``width`` values.

    The cheapest by an estimate in us: a walk of 0.75 per tile of 32 keys in bf16 and 2.8 in f32, once per 512 blocks, and with
    parts a second launch that reads them all.  Unsplit / in 2 / as chosen (window 1 << 30, 16 heads over 4): 8 prompts of 100 rows
    7.9 / 21.1 / 7.9, one of 1000 29 / 35 / 29, of 300 rows behind 600 beside 30 single rows 30.0 / 25.7 / 25.7, of 64 rows behind
    836 25.5 / 18.3 / 15.4; one row behind 1000 25.3 / 17.3 / 13.7, behind 100 6.7 / 7.9 / 6.7; in f32 8 of 100 17.6 / 27.4 / 17.6,
    one row behind 100 15.9 / 12.3 / 12.3."""
    tiles = (keys + 31) // 32 + 1
    walk, merge = 0.75 if dtype == torch.bfloat16 else 2.8, 1.84e-6 * pairs * (width + 2)

    def cost(n: int) -> float:
        return walk * tiles / n * max(1, -(-blocks * n // 512)) + (2.5 + 4e-4 * pairs + (merge + 0.5) * n if n > 1 else 0.0)
    return min(range(1, max(1, min(16, tiles // 2, most_blocks // max(blocks, 1))) + 1), key=cost)


def latent_attend(q_lat: torch.Tensor, q_rot: torch.Tensor, cache: torch.Tensor, cu: torch.Tensor, pos: torch.Tensor,
                  bt: torch.Tensor, window: int, scale: float, max_len: int,
                  gate: Optional[torch.Tensor] = None, sink: Optional[torch.Tensor] = None,
                  exact_weights: bool = False) -> torch.Tensor:
    """Windowed causal attention in the latent space.  ``q_lat`` [T, H, R], ``q_rot`` [T, H, Dr];
    cache rows [c | k_rot]; the query at position p sees the keys j of its own sequence with
    0 <= p - j < window; score = (q_lat . c_j + q_rot . k_rot_j) * scale, f32 softmax,
    out[t, h] = sum_j p_j c_j, times sigmoid(gate[t, h]) when a gate [T, H] is given.  ``sink`` (f32 [H]): the
    softmax denominator of head h also holds exp(sink[h]).  ``exact_weights``: the bf16 kernel multiplies the
    latents by the softmax weights as two bf16 terms instead of one (f32 kernels always use f32 weights)."""
    T, H, R = q_lat.shape
    Dr = q_rot.shape[2]
    S = cu.numel() - 1
    if sink is not None and (sink.dtype != torch.float32 or sink.numel() != H):
        raise ValueError("sink: one f32 value per query head")
    if N.use_native(q_lat):
        assert q_lat.is_contiguous() and q_rot.is_contiguous() and bt.is_contiguous()
        out = torch.empty((T, H, R), dtype=q_lat.dtype, device=q_lat.device)
        # steps whose blocks (64 pairs of a row and a head) would leave the chip idle may walk each row's keys with several
        # blocks; the split depends only on static sizes (graph-safe).  R = 256 (64 keys per tile, two blocks per CU; 32
        # heads, window 1024): 64 single rows take 24 us with 256 blocks, 42 with 1024
        nsplit, ws = 1, None
        tiled = R == 256 and Dr in (0, 32)
        if tiled or (q_lat.dtype == torch.bfloat16 and max_len == 1):
            keys = min(window + min(max_len, 64), bt.shape[1] * PAGE)      # a block's rows are 64 at most
            blocks = S * ((H + 63) // 64) if max_len == 1 else S + T * H // 64
            if tiled:
                nsplit = _key_parts(keys, blocks, 512 if max_len > 1 else 256, T * H, R, q_lat.dtype)
            else:
                nsplit = max(1, min(16, ((keys + 31) // 32 + 1) // 2, 1024 // max(blocks, 1)))
            if nsplit > 1:
                ws = torch.empty((T, H, nsplit, R + 2), dtype=torch.float32, device=q_lat.device)
        N.mcall("mx_latent_attend", N.ptr(q_lat), N.ptr(q_rot), N.ptr(cache), N.ptr(cu), N.ptr(pos), N.ptr(bt),
                bt.shape[1], N.ptr(_rows(gate)) if gate is not None else None,
                gate.stride(0) if gate is not None else 0, N.ptr(sink), 1 if exact_weights else 0,
                int(min(window, 1 << 30)), float(scale), N.ptr(out), _dt(q_lat), S, int(max_len), H, R, Dr, nsplit, N.ptr(ws), T, N.stream())
        return out
    out = torch.zeros((T, H, R), dtype=torch.float32)
    rows = cache.view(-1, R + Dr).float()
    cul, pl = cu.tolist(), pos.tolist()
    for s in range(S):
        a, b = cul[s], cul[s + 1]
        if b <= a:
            continue
        ctx = pl[b - 1] + 1
        pages = bt[s, :(ctx + PAGE - 1) // PAGE].long()
        keys = rows.view(-1, PAGE, R + Dr)[pages].reshape(-1, R + Dr)[:ctx]
        qq = torch.cat([q_lat[a:b].float(), q_rot[a:b].float()], -1)       # [n, H, D]
        sc = torch.einsum("nhd,jd->nhj", qq, keys) * scale
        p = pos[a:b].long()[:, None]
        j = torch.arange(ctx)[None]
        vis = (j <= p) & (j > p - window)
        sc = sc.masked_fill(~vis[:, None, :], float("-inf"))
        out[a:b] = torch.einsum("nhj,jr->nhr", _sink_softmax(sc, sink), keys[:, :R])
    if gate is not None:
        out = out * torch.sigmoid(gate.float())[:, :, None]
    return out.to(q_lat.dtype)


# ----------------------------------------------------------------------------------------------
# sequential (post-norm) blocks: hashed pair embedding, layer norm on the sublayer output
# ----------------------------------------------------------------------------------------------
def embed_pairs(ids: torch.Tensor, table: torch.Tensor, pair_table: Optional[torch.Tensor], mul_prev: int, mul_cur: int,
                last_token: Optional[torch.Tensor], cu: torch.Tensor, slot: torch.Tensor, pos: torch.Tensor,
                max_len: int) -> torch.Tensor:
    """f32 residual stream [T, W]: ``table[id]`` plus, with a ``pair_table`` [buckets + 1, W], its row
    ``(prev * mul_prev + id * mul_cur) mod buckets`` -- ``prev`` the token before in the same
    sequence -- or row ``buckets`` at position 0.  ``last_token`` int32 [slots] holds every slot's
    last token between steps (read by a segment's first row, then replaced by its last id)."""
    T, (V, W) = ids.numel(), table.shape
    S = cu.numel() - 1
    ids = ids.to(torch.int32).contiguous()
    if pair_table is None:
        return embed_f32(ids, table)
    B = pair_table.shape[0] - 1
    if N.use_native(table):
        out = torch.empty((T, W), dtype=torch.float32, device=table.device)
        N.mcall("mx_embed_pairs", N.ptr(ids), N.ptr(table), N.ptr(pair_table), _dt(table), int(mul_prev), int(mul_cur),
                B, N.ptr(last_token), N.ptr(cu), N.ptr(slot), N.ptr(pos), N.ptr(out), S, int(max_len), W, V, N.stream())
        return out
    out = table[ids.long().clamp(0, V - 1)].float()
    cul, sll, pl, idl = cu.tolist(), slot.tolist(), pos.tolist(), ids.tolist()
    for s in range(S):
        a, b = cul[s], cul[s + 1]
        if sll[s] < 0 or b <= a:
            continue
        for r in range(a, b):
            if pl[r] == 0:
                row = B
            else:
                prev = idl[r - 1] if r > a else int(last_token[sll[s]])
                row = (prev * mul_prev + idl[r] * mul_cur) % B
            out[r] += pair_table[row].float()
        last_token[sll[s]] = idl[b - 1]
    return out


def _ln(v: torch.Tensor, w: torch.Tensor, eps: float) -> torch.Tensor:
    mu = v.mean(-1, keepdim=True)
    d = v - mu
    return d * torch.rsqrt(d.pow(2).mean(-1, keepdim=True) + eps) * w.float()


def layer_norm_out(x: torch.Tensor, w: torch.Tensor, eps: float, out_dtype: torch.dtype) -> torch.Tensor:
    """(x - mean) / sqrt(var + eps) * w of every f32 row, in ``out_dtype``."""
    T, W = x.shape
    assert x.dtype == torch.float32 and x.is_contiguous()
    if N.use_native(x):
        out = torch.empty((T, W), dtype=out_dtype, device=x.device)
        N.mcall("mx_post_norm", N.ptr(x), None, 0, None, None, 0, None, 1, N.ptr(w), float(eps), N.ptr(out), _dt(out),
                T, W, N.stream())
        return out
    return _ln(x, w, eps).to(out_dtype)


def post_norm_add(x: torch.Tensor, a: Sublayer, w: torch.Tensor, eps: float, out_dtype: Optional[torch.dtype] = None,
                  b: Optional[Sublayer] = None, wa: Optional[torch.Tensor] = None,
                  wb: Optional[torch.Tensor] = None) -> Optional[torch.Tensor]:
    """``x`` (f32 [T, W], in place) <- x + LayerNorm(m) * w, the norm on the sublayer's output only.
    m = a, or with a second branch m = (RMSnorm(a) * wa + RMSnorm(b) * wb) / 2 (two mixers side by
    side).  Returns the new x rounded to ``out_dtype`` (the next sublayer's GEMM input) when one is
    given and differs from f32, else x itself."""
    T, W = x.shape
    assert x.dtype == torch.float32 and x.is_contiguous()
    want = out_dtype is not None and out_dtype != torch.float32
    parts = _parts(x, a, b, 4096) if (w.data_ptr() | (N.ptr(wa) or 0) | (N.ptr(wb) or 0)) % 16 == 0 else None
    if parts is not None:
        out = torch.empty((T, W), dtype=out_dtype, device=x.device) if want else None
        N.mcall("mx_post_norm_parts", N.ptr(x), parts[0], N.ptr(wa), parts[1], N.ptr(wb), int(a.dtype == torch.float32), N.ptr(w), float(eps),
                N.ptr(out), _dt(out) if want else 1, T, W, N.stream())
        return out if want else x
    a, b = whole(a), whole(b)
    if N.use_native(x):
        out = torch.empty((T, W), dtype=out_dtype, device=x.device) if want else None
        if b is not None:
            assert a.dtype == b.dtype
        N.mcall("mx_post_norm", N.ptr(x), N.ptr(_rows(a)), a.stride(0), N.ptr(wa), N.ptr(_rows(b)) if b is not None else None,
                b.stride(0) if b is not None else 0, N.ptr(wb), _dt(a), N.ptr(w), float(eps), N.ptr(out),
                _dt(out) if want else 1, T, W, N.stream())
        return out if want else x
    m = a.float()
    if b is not None:
        rms = lambda v: v * torch.rsqrt(v.pow(2).mean(-1, keepdim=True) + eps)  # noqa: E731
        m = 0.5 * (rms(m) * wa.float() + rms(b.float()) * wb.float())
    x.add_(_ln(m, w, eps))
    return x.to(out_dtype) if want else x


ACTS = {"none": 0, "silu": 1, "gelu_tanh": 2, "sigmoid": 3}


def _act(v: torch.Tensor, act: str) -> torch.Tensor:
    if act == "silu":
        return F.silu(v)
    if act == "gelu_tanh":
        return F.gelu(v, approximate="tanh")
    if act == "sigmoid":
        return torch.sigmoid(v)
    return v


def glu_act(gate: torch.Tensor, up: Optional[torch.Tensor], act: str,
            row_scale: Optional[torch.Tensor] = None) -> torch.Tensor:
    """act(s * gate) * (s * up) with ``s`` an optional f32 scale per row (a routed expert whose weight
    multiplies its INPUT: the scale commutes with the two projections); ``act``: silu | gelu_tanh | sigmoid.
    ``up`` None: act(s * gate) alone (a plain, ungated feed-forward)."""
    T, n = gate.shape
    if N.use_native(gate):
        out = torch.empty((T, n), dtype=gate.dtype, device=gate.device)
        N.mcall("mx_glu_act", N.ptr(_rows(gate)), gate.stride(0), N.ptr(_rows(up)) if up is not None else None,
                up.stride(0) if up is not None else 0, N.ptr(row_scale), ACTS[act], N.ptr(out), out.stride(0), _dt(gate),
                T, n, N.stream())
        return out
    g = gate.float()
    if row_scale is not None:
        g = g * row_scale[:, None]
    if up is None:
        return _act(g, act).to(gate.dtype)
    u = up.float() * (row_scale[:, None] if row_scale is not None else 1.0)
    return (_act(g, act) * u).to(gate.dtype)


ROUTE_SCORES = {"softmax": 0, "sigmoid": 1, "softmax_top": 2}


def route_scores(z: torch.Tensor, top: int, score: str = "sigmoid") -> Tuple[torch.Tensor, torch.Tensor]:
    """The ``top`` largest entries of each row of the f32 router logits ``z`` (ties: the lower index)
    and their scores: ``sigmoid`` (independent per expert) or ``softmax`` over all entries, neither
    renormalised, or ``softmax_top``: the softmax over the chosen logits only.
    Returns (weights f32 [T, top], indices int32 [T, top]), the largest first."""
    T, E = z.shape
    assert z.dtype == torch.float32
    if N.use_native(z):
        z = z.contiguous()
        w = torch.empty((T, top), dtype=torch.float32, device=z.device)
        i = torch.empty((T, top), dtype=torch.int32, device=z.device)
        N.mcall("mx_route_scores", N.ptr(z), E, top, ROUTE_SCORES[score], N.ptr(w), N.ptr(i), T, N.stream())
        return w, i
    if score == "softmax_top":
        # a stable sort: ties go to the lower index, as in the kernel
        idx = torch.sort(z, dim=-1, descending=True, stable=True).indices[:, :top]
        return torch.softmax(z.gather(1, idx), -1), idx.to(torch.int32)
    if score not in ROUTE_SCORES:
        raise ValueError(f"unknown routing score {score!r}")
    s = torch.sigmoid(z) if score == "sigmoid" else torch.softmax(z, -1)
    idx = torch.topk(s, top, dim=-1).indices
    return s.gather(1, idx), idx.to(torch.int32)


def conv_act(inp: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor], state: torch.Tensor, cu: torch.Tensor,
             slot: torch.Tensor, pos: torch.Tensor, max_len: int, act: str = "silu",
             in_bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """:func:`conv_silu` with the activation as a parameter (``silu`` | ``none``) and an optional
    bias ``in_bias`` [C] added to every input BEFORE the convolution (inputs before the sequence stay
    zero; the slot's history holds biased inputs)."""
    if act == "silu" and in_bias is None:
        return conv_silu(inp, w, bias, state, cu, slot, pos, max_len)
    T, C = inp.shape
    K = w.shape[1]
    S = cu.numel() - 1
    if N.use_native(inp):
        out = torch.empty((T, C), dtype=torch.float32, device=inp.device)
        N.mcall("mx_conv_act", N.ptr(_rows(inp)), inp.stride(0), _dt(inp), N.ptr(w), N.ptr(bias), N.ptr(in_bias),
                ACTS[act], N.ptr(state), N.ptr(cu), N.ptr(slot), N.ptr(pos), N.ptr(out), S, int(max_len), T, C, K, N.stream())
        return out
    out = torch.zeros((T, C), dtype=torch.float32)
    cul, sll, pl = cu.tolist(), slot.tolist(), pos.tolist()
    x = inp.float() + (in_bias.float() if in_bias is not None else 0.0)
    for s in range(S):
        a, b = cul[s], cul[s + 1]
        if sll[s] < 0 or b <= a:
            continue
        hist = torch.zeros((K - 1, C)) if pl[a] == 0 else state[sll[s]].clone()
        full = torch.cat([hist, x[a:b]])
        acc = (full.unfold(0, K, 1) * w.float()[None]).sum(-1)
        if bias is not None:
            acc = acc + bias.float()
        out[a:b] = _act(acc, act)
        if K > 1:
            state[sll[s]] = full[-(K - 1):]
    return out


# ----------------------------------------------------------------------------------------------
# matrix-state linear recurrences (gated linear attention, gated delta rule)
# ----------------------------------------------------------------------------------------------
SCAN_CHUNK_LEAST = 32         # the longest segment from which the chunk form is possible (SCAN_LEAST of the kernels)


def matrix_scan(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, a: torch.Tensor, a_bias: torch.Tensor,
                state: torch.Tensor, cu: torch.Tensor, slot: torch.Tensor, pos: torch.Tensor, heads: int, kv_heads: int,
                dim: int, vdim: int, mode: str, tau: float = 1.0, A_log: Optional[torch.Tensor] = None,
                beta: Optional[torch.Tensor] = None, max_len: int = 0) -> torch.Tensor:
    """Token-by-token f32 recurrence over a [dim, vdim] state per head (``state`` f32
    [slots, H, dim, vdim], read unless the segment starts at position 0, then replaced), with one
    decay per head and key channel acting on the state's rows.  ``q``/``k`` [T, G*dim], ``v``
    [T, H*vdim] (column slices; head h reads q/k head h // (H/G)), ``a`` f32 [T, H*dim] the decay's
    pre-activation (the kernels may overwrite it with the decays), ``a_bias`` f32 [H*dim].

    ``mode="gla"``:   g = sigmoid(a + a_bias)^(1/tau);  S <- g S + k v^T;  o = S^T (q dim^-1/2).
    ``mode="delta"``: q, k <- unit vectors (x / sqrt(sum x^2 + 1e-6)), q scaled by dim^-1/2;
                      g = exp(-exp(A_log[h]) softplus(a + a_bias));  b = sigmoid(beta[t, h]);
                      S <- g S;  u = b (v - S^T k);  S <- S + k u^T;  o = S^T q.
    ``max_len``: the longest segment when known (1 selects the kernels' single-row form, left out the token form).
    Returns o f32 [T, H*vdim]."""
    T = q.shape[0]
    H, G, D, P = heads, kv_heads, dim, vdim
    S = cu.numel() - 1
    delta = mode == "delta"
    assert a.dtype == torch.float32 and a.shape[1] == H * D and q.shape[1] == G * D and v.shape[1] == H * P
    assert q.dtype == k.dtype == v.dtype
    if N.use_native(q):
        out = torch.empty((T, H * P), dtype=torch.float32, device=q.device)
        aux = torch.empty((T, 2 * G + H), dtype=torch.float32, device=q.device) if delta else None
        ws = None
        if max_len >= SCAN_CHUNK_LEAST and D <= 256:
            DP = 64 if D <= 64 else 128 if D <= 128 else 256
            ws = torch.empty((T // 16 + S, H, 33 * DP + 256 + (16 * DP + 256 if delta else 0)), dtype=torch.float32, device=q.device)
        N.mcall("mx_matrix_scan", N.ptr(_rows(q)), q.stride(0), N.ptr(_rows(k)), k.stride(0), N.ptr(_rows(v)), v.stride(0),
                _dt(q), N.ptr(_rows(a)), a.stride(0), N.ptr(a_bias), N.ptr(A_log) if delta else None,
                N.ptr(_rows(beta)) if delta else None, beta.stride(0) if delta else 0, _dt(beta) if delta else 1,
                float(tau), 1 if delta else 0, N.ptr(aux), N.ptr(ws), N.ptr(state), N.ptr(cu), N.ptr(slot), N.ptr(pos), N.ptr(out), S, T,
                int(max_len), H, G, D, P, N.stream())
        return out
    out = torch.zeros((T, H * P), dtype=torch.float32)
    cul, sll, pl = cu.tolist(), slot.tolist(), pos.tolist()
    rep = H // G
    for s in range(S):
        r0, r1 = cul[s], cul[s + 1]
        if sll[s] < 0 or r1 <= r0:
            continue
        n = r1 - r0
        qq = q[r0:r1].float().view(n, G, D)
        kk = k[r0:r1].float().view(n, G, D)
        vv = v[r0:r1].float().view(n, H, P)
        z = a[r0:r1].float() + a_bias.float()
        if delta:
            qq = qq * torch.rsqrt(qq.pow(2).sum(-1, keepdim=True) + 1e-6)
            kk = kk * torch.rsqrt(kk.pow(2).sum(-1, keepdim=True) + 1e-6)
            g = torch.exp(-torch.exp(A_log.float()).repeat_interleave(D)[None] * F.softplus(z)).view(n, H, D)
            bt = torch.sigmoid(beta[r0:r1].float())
        else:
            g = torch.exp(-F.softplus(-z) / tau).view(n, H, D)
        qq = (qq * D ** -0.5).repeat_interleave(rep, 1)
        kk = kk.repeat_interleave(rep, 1)
        St = torch.zeros((H, D, P)) if pl[r0] == 0 else state[sll[s]].clone()
        for t in range(n):
            St = g[t][:, :, None] * St
            u = vv[t]
            if delta:
                u = bt[t][:, None] * (u - torch.einsum("hdp,hd->hp", St, kk[t]))
            St = St + kk[t][:, :, None] * u[:, None, :]
            out[r0 + t] = torch.einsum("hdp,hd->hp", St, qq[t]).reshape(-1)
        state[sll[s]] = St
    return out


def low_rank(ua: torch.Tensor, wa: torch.Tensor, ug: Optional[torch.Tensor] = None,
             wg: Optional[torch.Tensor] = None) -> Tuple[torch.Tensor, Optional[torch.Tensor]]:
    """The second factors of two low-rank projections: ``ua wa^T`` in f32 (``ua`` [T, ra] bf16 or f32, ``wa`` f32) and, given, ``ug wg^T`` in
    the type of ``ug``.  One launch for ranks of 32 and 64 (``mx_low_rank``), else, and under autocast or for gradients, a product each."""
    (T, ra), na = ua.shape, wa.shape[0]
    plain = not torch.is_autocast_enabled() and not any(t is not None and t.requires_grad for t in (ua, wa, ug, wg))
    if plain and N.use_native(ua) and T > 0 and ra in (32, 64) and na % 16 == 0 and wa.dtype == torch.float32 and wa.shape[1] == ra and wa.is_contiguous() and \
            ua.dtype in (torch.bfloat16, torch.float32) and ua.stride(1) == 1 and ua.stride(0) * ua.element_size() % 16 == 0 and ua.stride(0) >= ra and \
            (ua.data_ptr() | wa.data_ptr()) % 16 == 0 and T <= 128 * 65535:
        ng = 0 if ug is None else wg.shape[0]
        if ng == 0 or (ug.shape[0] == T and ug.shape[1] in (32, 64) and ug.shape[1] <= ug.stride(0) and wg.shape[1] == ug.shape[1] and ng % 16 == 0 and ug.stride() == ua.stride() and
                       ug.dtype == wg.dtype == ua.dtype and wg.is_contiguous() and (ug.data_ptr() | wg.data_ptr()) % 16 == 0):
            a = torch.empty((T, na), dtype=torch.float32, device=ua.device)
            g = torch.empty((T, ng), dtype=ua.dtype, device=ua.device) if ng else None
            N.mcall("mx_low_rank", N.ptr(ua), N.ptr(ug), ua.stride(0), N.ptr(wa), ra, na, N.ptr(wg), ug.shape[1] if ng else 0, ng, N.ptr(a), N.ptr(g),
                    _dt(ua), T, N.stream())
            return a, g
    return project(ua.float(), wa), project(ug, wg) if ug is not None else None


def head_norm_gate(o: torch.Tensor, w: torch.Tensor, eps: float, gate: torch.Tensor, heads: int, act: str,
                   out_dtype: torch.dtype) -> torch.Tensor:
    """Every head's part of ``o`` [T, H*P] divided by its root mean square over P, times ``w`` [P]
    (shared by the heads; None: no weight), times act(gate) [T, H*P]; ``act``: sigmoid | silu.  With
    ``heads=1`` the whole row is normed at once with a weight per column."""
    T, n = o.shape
    P = n // heads
    if N.use_native(o):
        out = torch.empty((T, n), dtype=out_dtype, device=o.device)
        N.mcall("mx_head_norm_gate", N.ptr(_rows(o)), o.stride(0), _dt(o), N.ptr(w), float(eps), N.ptr(_rows(gate)),
                gate.stride(0), _dt(gate), ACTS[act], N.ptr(out), _dt(out), T, heads, P, N.stream())
        return out
    v = o.float().view(T, heads, P)
    v = v * torch.rsqrt(v.pow(2).mean(-1, keepdim=True) + eps)
    if w is not None:
        v = v * w.float()
    return (v.reshape(T, n) * _act(gate.float(), act)).to(out_dtype)


# ----------------------------------------------------------------------------------------------
# real-gated linear recurrent unit
# ----------------------------------------------------------------------------------------------
def lru_scan(u: torch.Tensor, z: torch.Tensor, blocks: int, r_bias: torch.Tensor, i_bias: torch.Tensor,
             lam: torch.Tensor, y: torch.Tensor, y_bias: Optional[torch.Tensor], state: torch.Tensor, cu: torch.Tensor,
             slot: torch.Tensor, pos: torch.Tensor, out_dtype: torch.dtype, max_len: int = 0) -> torch.Tensor:
    """Per channel, f32: r = sigmoid(zr + r_bias), i = sigmoid(zi + i_bias), a = exp(-8 r softplus(lam)),
    S <- a S + sqrt(1 - a^2) i u (also for a sequence's first token, from S = 0); returns
    S * gelu_tanh(y + y_bias) in ``out_dtype``.  ``u`` f32 [T, R] (the kernels reuse it as scratch);
    ``z`` f32 [blocks, T, 2 * R / blocks]:
    block b's gate pre-activations [zr | zi] as the batched block-diagonal product leaves them (the
    kernels overwrite it with the gates);
    ``y`` a column slice; ``state`` f32 [slots, R], read unless the segment starts at position 0,
    then replaced.  ``max_len``: the longest segment when known (1 selects the fused single-row kernel)."""
    T, R = u.shape
    S = cu.numel() - 1
    bs = R // blocks
    assert u.dtype == z.dtype == torch.float32 and u.is_contiguous() and z.is_contiguous()
    assert tuple(z.shape) == (blocks, T, 2 * bs)
    if N.use_native(u):
        out = torch.empty((T, R), dtype=out_dtype, device=u.device)
        N.mcall("mx_lru_scan", N.ptr(u), N.ptr(z), blocks, N.ptr(r_bias), N.ptr(i_bias), N.ptr(lam), N.ptr(_rows(y)),
                y.stride(0), _dt(y), N.ptr(y_bias), N.ptr(state), N.ptr(cu), N.ptr(slot), N.ptr(pos), N.ptr(out), _dt(out),
                S, R, T, int(max_len), N.stream())
        return out
    zr = z[:, :, :bs].transpose(0, 1).reshape(T, R)
    zi = z[:, :, bs:].transpose(0, 1).reshape(T, R)
    out = torch.zeros((T, R), dtype=torch.float32)
    cul, sll, pl = cu.tolist(), slot.tolist(), pos.tolist()
    a = torch.exp(-8.0 * torch.sigmoid(zr + r_bias.float()) * F.softplus(lam.float()))
    bx = torch.sqrt(1.0 - a * a) * torch.sigmoid(zi + i_bias.float()) * u
    yy = y.float() + (y_bias.float() if y_bias is not None else 0.0)
    for s in range(S):
        r0, r1 = cul[s], cul[s + 1]
        if sll[s] < 0 or r1 <= r0:
            continue
        St = torch.zeros(R) if pl[r0] == 0 else state[sll[s]].clone()
        for t in range(r0, r1):
            St = a[t] * St + bx[t]
            out[t] = St
        state[sll[s]] = St
    return (out * F.gelu(yy, approximate="tanh")).to(out_dtype)


def lru_blocks(u: torch.Tensor, w: torch.Tensor, r_bias: torch.Tensor, i_bias: torch.Tensor, lam: torch.Tensor, y: torch.Tensor,
               y_bias: Optional[torch.Tensor], state: torch.Tensor, cu: torch.Tensor, slot: torch.Tensor, pos: torch.Tensor,
               out_dtype: torch.dtype, max_len: int = 0) -> torch.Tensor:
    """:func:`lru_scan` from the block-diagonal gate matrices ``w`` f32 [blocks, 2 bs, bs] (r over i) of ``u`` f32 [T, blocks bs], which
    is scratch afterwards: product and gates in one launch for blocks in whole 64s, but for single-row steps.  Those keep the batched
    product, on this layout as on its transpose (us in a replayed graph, transpose / this: 8 blocks of 256, 1 row 4.2 / 4.0, 32 4.8 / 4.5, 64
    5.2 / 5.8, 128 6.8 / 6.0; 4 of 256, 64 4.7 / 6.4; 8 of 128, 1 6.0 / 6.4, 128 19.8 / 19.9; 10 of 256, 64 8.2 / 9.6, 128 14.8 / 8.9)."""
    T, R = u.shape
    B, bs = w.shape[0], w.shape[2]
    if N.use_native(u) and max_len != 1 and bs % 64 == 0 and 0 < T * R < 1 << 31 and R <= 64 * 65535 and cu.numel() <= 65535 and \
            u.is_contiguous() and w.is_contiguous() and (u.data_ptr() | w.data_ptr()) % 16 == 0:
        assert u.dtype == w.dtype == torch.float32 and tuple(w.shape) == (B, 2 * bs, bs) and R == B * bs
        z = torch.empty((B, T, 2 * bs), dtype=torch.float32, device=u.device)
        gy = torch.empty((T, R), dtype=torch.float32, device=u.device)
        out = torch.empty((T, R), dtype=out_dtype, device=u.device)
        N.mcall("mx_lru_blocks", N.ptr(u), N.ptr(w), B, N.ptr(r_bias), N.ptr(i_bias), N.ptr(lam), N.ptr(_rows(y)), y.stride(0), _dt(y),
                N.ptr(y_bias), N.ptr(z), N.ptr(gy), N.ptr(state), N.ptr(cu), N.ptr(slot), N.ptr(pos), N.ptr(out), _dt(out),
                cu.numel() - 1, R, T, N.stream())
        return out
    z = torch.bmm(u.view(T, B, bs).transpose(0, 1), w.transpose(1, 2))             # [B, T, 2 bs]: r | i pre-activations
    return lru_scan(u, z, B, r_bias, i_bias, lam, y, y_bias, state, cu, slot, pos, out_dtype, max_len=max_len)


# ----------------------------------------------------------------------------------------------
# minimal gated recurrent unit
# ----------------------------------------------------------------------------------------------
def mingru_scan(zp: torch.Tensor, xp: torch.Tensor, gp: torch.Tensor, z_bias: Optional[torch.Tensor],
                x_bias: Optional[torch.Tensor], state: torch.Tensor, cu: torch.Tensor, slot: torch.Tensor,
                pos: torch.Tensor, out_dtype: torch.dtype, max_len: int = 0) -> torch.Tensor:
    """Per channel, f32: z = sigmoid(zp + z_bias), u = xp + x_bias, candidate c = u + 1/2 where u >= 0 and
    sigmoid(u) below, S <- (1 - z) S + z c (gates from the current token only); returns S * silu(gp) in
    ``out_dtype``.  ``zp``, ``xp``, ``gp`` [T, R] are column slices of one projection; ``state`` f32
    [slots, R], read unless the segment starts at position 0, then replaced.  ``max_len``: the longest
    segment when known (1 selects the fused single-row kernel)."""
    T, R = zp.shape
    S = cu.numel() - 1
    assert xp.shape == zp.shape == gp.shape and zp.dtype == xp.dtype == gp.dtype
    if N.use_native(zp):
        out = torch.empty((T, R), dtype=out_dtype, device=zp.device)
        one = max_len == 1
        ab = None if one else torch.empty((T, 2 * R), dtype=torch.float32, device=zp.device)
        gy = None if one else torch.empty((T, R), dtype=torch.float32, device=zp.device)
        N.mcall("mx_mingru_scan", N.ptr(_rows(zp)), zp.stride(0), N.ptr(_rows(xp)), xp.stride(0), N.ptr(_rows(gp)),
                gp.stride(0), _dt(zp), N.ptr(z_bias), N.ptr(x_bias), N.ptr(ab), N.ptr(gy), N.ptr(state), N.ptr(cu),
                N.ptr(slot), N.ptr(pos), N.ptr(out), _dt(out), S, R, T, int(max_len), N.stream())
        return out
    a = zp.float() + (z_bias.float() if z_bias is not None else 0.0)
    u = xp.float() + (x_bias.float() if x_bias is not None else 0.0)
    keep, put = torch.sigmoid(-a), torch.sigmoid(a) * torch.where(u >= 0, u + 0.5, torch.sigmoid(u))
    out = torch.zeros((T, R), dtype=torch.float32)
    cul, sll, pl = cu.tolist(), slot.tolist(), pos.tolist()
    for s in range(S):
        r0, r1 = cul[s], cul[s + 1]
        if sll[s] < 0 or r1 <= r0:
            continue
        St = torch.zeros(R) if pl[r0] == 0 else state[sll[s]].clone()
        for t in range(r0, r1):
            St = keep[t] * St + put[t]
            out[t] = St
        state[sll[s]] = St
    return (out * F.silu(gp.float())).to(out_dtype)


# ----------------------------------------------------------------------------------------------
# sliding-window attention with grouped key/value heads over a paged row cache
# ----------------------------------------------------------------------------------------------
def qk_norm_write(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, qw: Optional[torch.Tensor],
                  kw: Optional[torch.Tensor], eps: float, slots: torch.Tensor, cache: torch.Tensor, dim: int = 0,
                  freq: Optional[torch.Tensor] = None, pos: Optional[torch.Tensor] = None, layout: str = "half",
                  mscale: float = 1.0) -> torch.Tensor:
    """Per token: RMS norm of the WHOLE query projection (all heads at once) times ``qw`` -> returned
    [T, nq]; the same for the key projection with ``kw``; the normed keys and the values go to cache
    row ``slots[t]`` as [k | v] (< 0: no write).  ``qw``/``kw`` None: no norm (without ``qw`` the returned
    queries are ``q`` itself, a column slice: nothing is copied).  With ``freq`` (f32 [rot / 2]) the first ``rot``
    entries of every head of ``dim`` entries are rotated after the norm by the angle pos * freq_i (f32), pairs as in
    :func:`rope_heads`, cos and sin times ``mscale``."""
    T, nq = q.shape
    nk, nv = k.shape[1], v.shape[1]
    assert cache.shape[-1] == nk + nv
    rot = 2 * freq.numel() if freq is not None else 0
    if rot and (layout not in ("half", "pairs") or rot > dim or nq % dim or nk % dim or pos is None):
        raise ValueError("qk_norm_write: whole heads of dim entries, rotated part <= dim, layout half | pairs")
    if N.use_native(q):
        assert q.dtype == k.dtype == v.dtype == cache.dtype
        out = torch.empty((T, nq), dtype=q.dtype, device=q.device) if qw is not None or rot else None
        N.mcall("mx_qk_norm_write", N.ptr(_rows(q)), q.stride(0), N.ptr(_rows(k)), k.stride(0), N.ptr(_rows(v)), v.stride(0),
                N.ptr(qw), N.ptr(kw), float(eps), int(dim), rot, 1 if layout == "half" else 0, N.ptr(freq), float(mscale),
                N.ptr(pos), N.ptr(slots), N.ptr(cache), N.ptr(out), _dt(q), T, nq, nk, nv, N.stream())
        return out if out is not None else q
    rms = lambda t, w: (t.float() * torch.rsqrt(t.float().pow(2).mean(-1, keepdim=True) + eps) * w.float()  # noqa: E731
                        if w is not None else t.float())
    ang = pos.float()[:, None] * freq.float()[None, :] if rot else None

    def done(t, w):
        t = rms(t, w)
        return _rotate_heads(t.reshape(T, -1, dim), ang, rot, layout == "half", mscale).reshape(T, -1) if rot else t

    rows = torch.cat([done(k, kw), v.float()], 1).to(cache.dtype)
    ok = slots >= 0
    cache.view(-1, nk + nv)[slots[ok].long()] = rows[ok]
    return done(q, qw).to(q.dtype) if qw is not None or rot else q


def conv_heads(proj: torch.Tensor, w: torch.Tensor, state: Optional[torch.Tensor], q_norm: Optional[torch.Tensor],
               k_norm: Optional[torch.Tensor], eps: float, cu: torch.Tensor, slot: torch.Tensor, pos: torch.Tensor,
               slots: torch.Tensor, cache: Optional[torch.Tensor], max_len: int, heads: int, kv_heads: int, dim: int,
               vdim: int, temp_coef: float = 0.0, temp_every: int = 1) -> torch.Tensor:
    """Projected heads up to attention.  ``proj`` [T, C] (a column slice) holds the channels q: H*dim | k: G*dim |
    v: G*vdim; every channel is convolved causally over its segment with ``w`` f32 [C, K] (last column: the current
    token's tap, no activation; ``state`` f32 [slots, K-1, C]: each slot's last K-1 inputs, read unless the
    segment starts at position 0, then replaced; unused for K = 1).  Then each q and k head is divided by its root
    mean square over ``dim`` and multiplied by ``q_norm`` / ``k_norm`` f32 [dim] (None: neither), q by
    1 + temp_coef * ln(floor((p + 1) / temp_every) + 1) at position p.  The finished k and the convolved v go to
    ``cache`` row ``slots[t]`` as [k | v] (< 0: no write); q is returned [T, H*dim].  ``kv_heads`` 0: queries
    only, no cache row (a layer that reads another layer's keys and values)."""
    T = proj.shape[0]
    H, G, D, P = heads, kv_heads, dim, vdim
    K = w.shape[1]
    C = (H + G) * D + G * P
    S = cu.numel() - 1
    assert w.dtype == torch.float32 and w.shape[0] == C and proj.shape[1] >= C
    assert K == 1 or (state is not None and tuple(state.shape[1:]) == (K - 1, C))
    assert G == 0 or cache.shape[-1] == G * (D + P)
    if N.use_native(proj):
        assert G == 0 or cache.dtype == proj.dtype
        out = torch.empty((T, H * D), dtype=proj.dtype, device=proj.device)
        N.mcall("mx_conv_heads", N.ptr(_rows(proj)), proj.stride(0), _dt(proj), N.ptr(w), K, N.ptr(state) if K > 1 else None,
                N.ptr(q_norm), N.ptr(k_norm), float(eps), float(temp_coef), int(temp_every), N.ptr(cu), N.ptr(slot),
                N.ptr(pos), N.ptr(slots), N.ptr(cache) if G else None, N.ptr(out), S, int(max_len), T, H, G, D, P, N.stream())
        return out
    u = proj[:, :C].float()
    y = torch.zeros((T, C), dtype=torch.float32)
    cul, sll, pl = cu.tolist(), slot.tolist(), pos.tolist()
    for s in range(S):
        a, b = cul[s], cul[s + 1]
        if b <= a:
            continue
        old = K > 1 and sll[s] >= 0 and pl[a] != 0
        full = torch.cat([state[sll[s]] if old else torch.zeros((K - 1, C)), u[a:b]])
        y[a:b] = (full.unfold(0, K, 1) * w.float()[None]).sum(-1)
        if K > 1 and sll[s] >= 0:
            state[sll[s]] = full[-(K - 1):]

    def normed(t, nh, nw):
        t = t.reshape(T, nh, D)
        if nw is not None:
            t = t * torch.rsqrt(t.pow(2).mean(-1, keepdim=True) + eps) * nw.float()
        return t.reshape(T, nh * D)

    q = normed(y[:, :H * D], H, q_norm)
    if temp_coef:
        q = q * (1.0 + temp_coef * torch.log(((pos.long() + 1) // temp_every + 1).float()))[:, None]
    if G:
        rows = torch.cat([normed(y[:, H * D:(H + G) * D], G, k_norm), y[:, (H + G) * D:]], 1).to(cache.dtype)
        ok = slots >= 0
        cache.view(-1, G * (D + P))[slots[ok].long()] = rows[ok]
    return q.to(proj.dtype)


def distance_buckets(rows: int, far: float) -> torch.Tensor:
    """Row of a ``rows``-row bias table for every distance 0 .. L - 1 (int64; L - 1 is the first distance of the last
    row, which every larger distance shares): distance n itself below rows/2, from there in logarithmic steps that
    reach the last row before ``far``: rows/2 + floor(ln(n / (rows/2)) / ln(far / (rows/2)) * (rows - rows/2))."""
    import math
    half = rows // 2
    if half < 1 or not far > half:
        raise ValueError("distance buckets: at least two rows and far > rows / 2")
    out, n = list(range(half)), half
    while out[-1] < rows - 1:
        r = math.log(n / half) / math.log(far / half) * (rows - half)
        if abs(r - round(r)) < 1e-9:         # a step that falls on a whole distance is not left to rounding
            r = round(r)
        out.append(min(rows - 1, half + math.floor(r)))
        n += 1
    return torch.tensor(out, dtype=torch.int64)


def window_attend(q: torch.Tensor, cache: torch.Tensor, cu: torch.Tensor, pos: torch.Tensor, bt: torch.Tensor,
                  window: int, scale: float, max_len: int, heads: int, kv_heads: int, dim: int, vdim: int,
                  gate: Optional[torch.Tensor] = None, chunked: bool = False, keep_first: int = 0,
                  head_bias: Optional[torch.Tensor] = None, slopes: Optional[torch.Tensor] = None,
                  sink: Optional[torch.Tensor] = None, rel: Optional[torch.Tensor] = None,
                  softcap: float = 0.0) -> torch.Tensor:
    """Causal softmax attention of ``q`` [T, H*dim] over the cache rows [k: G*dim | v: G*vdim] of each
    segment's pages: the query at position p sees keys j with 0 <= p - j < window, or -- ``chunked`` --
    the keys j <= p with floor(j / window) == floor(p / window) (blocks of ``window`` positions counted
    from the start of the sequence); with ``keep_first`` the keys j < keep_first of the sequence stay
    visible to every later query as well (at their true positions).  Query head h
    reads key/value head h // (H/G); score = q . k * scale, f32 softmax -- or, with ``head_bias`` (f32 [H]),
    no softmax: the weight of a visible key is sigmoid(score + head_bias[h]), not normalised over the keys.
    ``softcap`` > 0: the scaled score becomes softcap * tanh(score / softcap) before any bias.  ``slopes`` (f32 [H]): a
    distance bias, slopes[h] * (p - j) is taken off the score; ``rel`` (f32 [H, L]): another, rel[h, min(p - j, L - 1)]
    is added to it.  ``sink`` (f32 [H],
    softmax only): the denominator of head h also holds exp(sink[h]).  Head h's output is multiplied by
    sigmoid(gate[t, h]) when a gate [T, H] is given, or element by element by sigmoid(gate) when the gate is
    [T, H*vdim].  Returns [T, H*vdim]."""
    T = q.shape[0]
    H, G, D, P = heads, kv_heads, dim, vdim
    S = cu.numel() - 1
    Wr = G * (D + P)
    for name, t in (("head_bias", head_bias), ("slopes", slopes), ("sink", sink)):
        if t is not None and (t.dtype != torch.float32 or t.numel() != H):
            raise ValueError(f"{name}: one f32 value per query head")
    if sink is not None and head_bias is not None:
        raise ValueError("a sink belongs to the softmax denominator; sigmoid weights have none")
    if rel is not None and (rel.dtype != torch.float32 or rel.dim() != 2 or rel.shape[0] != H or not rel.is_contiguous()):
        raise ValueError("rel: a contiguous f32 table [heads, distances]")
    if gate is not None and gate.shape[1] not in (H, H * P):
        raise ValueError("gate: one value per head or per output element")
    gate_elem = gate is not None and P > 1 and gate.shape[1] == H * P
    if N.use_native(q):
        assert bt.is_contiguous() and q.dtype == cache.dtype
        out = torch.empty((T, H * P), dtype=q.dtype, device=q.device)
        # steps whose blocks (64 pairs of a row and a head of one group) would leave the chip idle may walk each row's keys with
        # several blocks; the split depends only on static sizes (graph-safe).  Single rows may take 1024 blocks (48 rows of 16
        # heads over 4, window 1024: 25 us, at 256 blocks 39); with longer segments merging the parts costs more, and 512
        # are enough (577 rows in f32: 34 us at 468 blocks)
        nsplit, ws = 1, None
        tiled = D == 128 and P == 128 and head_bias is None and rel is None
        if tiled or (max_len == 1 and q.dtype == torch.bfloat16):
            keys = min(window + keep_first + min(max_len, 64), bt.shape[1] * PAGE)     # a block's rows are 64 at most
            blocks = S * G if max_len == 1 else (S + T * (H // G) // 64) * G
            most = 1024 if max_len == 1 else 512
            if tiled:
                nsplit = _key_parts(keys, blocks, most, T * H, P, q.dtype)
            else:
                nsplit = max(1, min(16, ((keys + 31) // 32 + 1) // 2, most // max(blocks, 1)))
            if nsplit > 1:
                ws = torch.empty((T, H, nsplit, P + 2), dtype=torch.float32, device=q.device)
        N.mcall("mx_window_attend", N.ptr(_rows(q)), q.stride(0), N.ptr(cache), N.ptr(cu), N.ptr(pos), N.ptr(bt), bt.shape[1],
                N.ptr(_rows(gate)) if gate is not None else None, gate.stride(0) if gate is not None else 0,
                1 if gate_elem else 0, int(min(window, 1 << 30)), 1 if chunked else 0, int(keep_first), N.ptr(head_bias),
                N.ptr(slopes), N.ptr(rel), rel.shape[1] if rel is not None else 0, float(softcap), N.ptr(sink), float(scale),
                N.ptr(out),
                _dt(q), S, int(max_len), H, G, D, P, nsplit, N.ptr(ws), T, N.stream())
        return out
    out = torch.zeros((T, H, P), dtype=torch.float32)
    rows = cache.view(-1, Wr).float()
    cul, pl = cu.tolist(), pos.tolist()
    rep = H // G
    for s in range(S):
        a, b = cul[s], cul[s + 1]
        if b <= a:
            continue
        ctx = pl[b - 1] + 1
        pages = bt[s, :(ctx + PAGE - 1) // PAGE].long()
        kv = rows.view(-1, PAGE, Wr)[pages].reshape(-1, Wr)[:ctx]
        keys = kv[:, :G * D].view(ctx, G, D).repeat_interleave(rep, 1)
        vals = kv[:, G * D:].view(ctx, G, P).repeat_interleave(rep, 1)
        sc = torch.einsum("nhd,jhd->nhj", q[a:b].float().view(-1, H, D), keys) * scale
        p = pos[a:b].long()[:, None]
        j = torch.arange(ctx)[None]
        if softcap > 0:
            sc = softcap * torch.tanh(sc / softcap)
        if rel is not None:
            sc = sc + rel[:, (p - j).clamp(0, rel.shape[1] - 1)].transpose(0, 1)
        if slopes is not None:
            sc = sc - slopes.float()[None, :, None] * (p - j).float()[:, None, :]
        vis = (j <= p) & (((j // window == p // window) if chunked else (j > p - window)) | (j < keep_first))
        if head_bias is not None:
            wt = torch.sigmoid(sc + head_bias.float()[None, :, None]) * vis[:, None, :]
        else:
            sc = sc.masked_fill(~vis[:, None, :], float("-inf"))
            wt = _sink_softmax(sc, sink)
        out[a:b] = torch.einsum("nhj,jhp->nhp", wt, vals)
    if gate is not None:
        out = out * torch.sigmoid(gate.float()).view(T, H, P if gate_elem else 1)
    return out.reshape(T, H * P).to(q.dtype)


# ----------------------------------------------------------------------------------------------
# several residual streams per token (hyper-connections); logit scale and soft cap
# ----------------------------------------------------------------------------------------------
MAX_STREAMS = 16


def embed_scaled(ids: torch.Tensor, table: torch.Tensor, scale: float = 1.0, copies: int = 1) -> torch.Tensor:
    """``copies`` equal f32 streams [T, copies, W] of ``table[id] * scale``."""
    T, (V, W) = ids.numel(), table.shape
    if N.use_native(table):
        out = torch.empty((T, copies, W), dtype=torch.float32, device=table.device)
        N.mcall("mx_embed_scaled", N.ptr(ids.to(torch.int32).contiguous()), N.ptr(table), _dt(table), float(scale),
                int(copies), N.ptr(out), T, W, V, N.stream())
        return out
    row = table[ids.long().clamp(0, V - 1)].float() * scale
    return row[:, None, :].repeat(1, copies, 1).contiguous()


def hyper_mix(x: torch.Tensor, y: Optional[torch.Tensor], mix: Optional[torch.Tensor], w_out: Optional[torch.Tensor],
              w_in: torch.Tensor, w: Optional[torch.Tensor], eps: float,
              out_dtype: torch.dtype = torch.bfloat16) -> Optional[torch.Tensor]:
    """One pass over the streams ``x`` (f32 [T, S, W], in place) between two sublayers.  With the output
    ``y`` [T, W] of the sublayer that just ran: x_t <- sum_s mix[s, t] x_s + w_out[t] * y for every
    stream t at once (``mix`` f32 [S, S] indexed [from, to], ``w_out`` f32 [S]).  Then the next
    sublayer's input u = sum_t w_in[t] x_t and its RMS norm u / sqrt(mean(u^2) + eps) * w in
    ``out_dtype`` (``w`` None: the update only).  S = 1 with mix = w_out = w_in = 1 is the plain
    pre-norm residual sum."""
    T, S, W = x.shape
    assert x.dtype == torch.float32 and x.is_contiguous()
    if S > MAX_STREAMS:
        raise ValueError(f"at most {MAX_STREAMS} residual streams are supported, got {S}")
    if N.use_native(x):
        out = torch.empty((T, W), dtype=out_dtype, device=x.device) if w is not None else None
        N.mcall("mx_hyper_mix", N.ptr(x), N.ptr(_rows(y)) if y is not None else None, y.stride(0) if y is not None else 0,
                _dt(y) if y is not None else 1, N.ptr(mix), N.ptr(w_out), N.ptr(w_in), N.ptr(w), float(eps), N.ptr(out),
                _dt(out) if out is not None else 1, T, S, W, N.stream())
        return out
    if y is not None:
        new = torch.einsum("st,nsw->ntw", mix.float(), x) + w_out.float()[None, :, None] * y.float()[:, None, :]
        x.copy_(new)
    if w is None:
        return None
    u = torch.einsum("t,ntw->nw", w_in.float(), x)
    return (u * torch.rsqrt(u.pow(2).mean(-1, keepdim=True) + eps) * w.float()).to(out_dtype)


def logit_cap(logits: torch.Tensor, scale: float = 1.0, cap: float = 0.0) -> torch.Tensor:
    """``logits`` <- cap * tanh(logits * scale / cap) in place (``cap`` <= 0: the scale only)."""
    if scale == 1.0 and cap <= 0:
        return logits
    if N.use_native(logits):
        assert logits.is_contiguous()
        N.mcall("mx_logit_cap", N.ptr(logits), _dt(logits), float(scale), float(cap), logits.numel(), N.stream())
        return logits
    v = logits.float() * scale
    if cap > 0:
        v = cap * torch.tanh(v / cap)
    return logits.copy_(v.to(logits.dtype))


# ----------------------------------------------------------------------------------------------
# rotation of projected heads
# ----------------------------------------------------------------------------------------------
def rope_freqs(dims: int, base: float, scaling: Optional[dict] = None, device=None) -> Tuple[torch.Tensor, float]:
    """Frequencies f_i = base^(-2i / dims), i < dims / 2 (f32) and the factor on cos and sin.  With a
    ``scaling`` entry {factor, original, fast, slow} (YaRN): with turn(t) = dims ln(original / (2 pi t)) /
    (2 ln base), lo = max(floor(turn(fast)), 0), hi = min(ceil(turn(slow)), dims - 1) and
    ramp_i = clamp((i - lo) / max(hi - lo, 0.001), 0, 1) the frequency is f_i / factor * ramp_i +
    f_i (1 - ramp_i) and cos and sin are multiplied by 0.1 ln(factor) + 1.  With {factor, original, low, high}
    (scaling by wavelength l = 2 pi / f): f is kept where l < original / high, divided by the factor where
    l > original / low, and (1 - s) f / factor + s f with s = (original / l - low) / (high - low) between.  A ``scaling`` entry with a factor
    only is linear scaling: every f_i is divided by the factor (positions are stretched), cos and sin unscaled."""
    import math
    i = torch.arange(dims // 2, dtype=torch.float64)
    f = float(base) ** (-2.0 * i / dims)
    m = 1.0
    if scaling and "original" not in scaling:      # linear scaling: every frequency divided by the factor
        f = f / float(scaling["factor"])
    elif scaling and "high" in scaling:
        factor, orig = float(scaling["factor"]), float(scaling["original"])
        low, high = float(scaling["low"]), float(scaling["high"])
        wave = 2 * math.pi / f
        s = (orig / wave - low) / (high - low) if high != low else torch.zeros_like(f)
        blend = (1 - s) * f / factor + s * f
        f = torch.where(wave < orig / high, f, torch.where(wave > orig / low, f / factor, blend))
    elif scaling:
        factor, orig = float(scaling["factor"]), float(scaling["original"])
        turn = lambda t: dims * math.log(orig / (2 * math.pi * float(t))) / (2 * math.log(float(base)))  # noqa: E731
        lo = max(math.floor(turn(scaling["fast"])), 0)
        hi = min(math.ceil(turn(scaling["slow"])), dims - 1)
        ramp = ((i - lo) / max(hi - lo, 0.001)).clamp(0, 1)
        f = f / factor * ramp + f * (1 - ramp)
        m = 0.1 * math.log(factor) + 1.0
    return f.to(torch.float32).to(device).contiguous(), m


def _rotate_heads(x: torch.Tensor, ang: torch.Tensor, rot: int, half: bool, m: float) -> torch.Tensor:
    """x f32 [T, H, D]; ang f32 [T, rot / 2]."""
    if rot == 0:
        return x
    c, s = (torch.cos(ang) * m)[:, None, :], (torch.sin(ang) * m)[:, None, :]
    out = x.clone()
    if half:
        a, b = x[..., :rot // 2], x[..., rot // 2:rot]
        out[..., :rot // 2] = a * c - b * s
        out[..., rot // 2:rot] = b * c + a * s
    else:
        a, b = x[..., 0:rot:2], x[..., 1:rot:2]
        out[..., 0:rot:2] = a * c - b * s
        out[..., 1:rot:2] = b * c + a * s
    return out


def rope_heads(q: torch.Tensor, k: torch.Tensor, heads: int, kv_heads: int, dim: int, freq: Optional[torch.Tensor],
               pos: torch.Tensor, layout: str = "pairs", mscale: float = 1.0, norm_eps: Optional[float] = None,
               q_scale: float = 1.0, k_scale: float = 1.0, q_dtype: Optional[torch.dtype] = None,
               k_out: Optional[torch.Tensor] = None, slots: Optional[torch.Tensor] = None,
               v: Optional[torch.Tensor] = None, k_dtype: Optional[torch.dtype] = None,
               v_mix: Optional[torch.Tensor] = None, v_lam: float = 0.0):
    """Per head of ``q`` [T, H*dim] and ``k`` [T, G*dim] (column slices): the first ``2 * len(freq)``
    entries are rotated by the angle pos * freq_i (f32), pair i being entries (2i, 2i+1) for
    ``layout="pairs"`` or (i, i + rot/2) for ``"half"``; (u, v) -> (u cos - v sin, v cos + u sin) with cos and
    sin times ``mscale``; then, with ``norm_eps``, the head is divided by its root mean square over
    ``dim`` (no weight); then times ``q_scale`` / ``k_scale``.  Returns (q', k'): q' [T, H*dim] in
    ``q_dtype``; k' [T, G*dim] in ``k_dtype`` -- or, with ``k_out`` (paged cache rows [rows, G*dim + nv])
    and ``slots`` [T], k' is written to row slots[t] (< 0: no write) followed by the raw values ``v``
    [T, nv], and None is returned for it; with ``v_mix`` ([T, nv]) the values written are
    (1 - v_lam) v + v_lam v_mix, blended in f32."""
    T = q.shape[0]
    H, G, D = heads, kv_heads, dim
    rot = 2 * freq.numel() if freq is not None else 0
    half = layout == "half"
    if layout not in ("pairs", "half") or rot > D:
        raise ValueError("rope_heads: layout is pairs | half and the rotated part must fit the head")
    q_dtype = q_dtype or q.dtype
    norm = norm_eps is not None
    if N.use_native(q):
        assert q.dtype == k.dtype and (v is None or v.dtype == q.dtype)
        qo = torch.empty((T, H * D), dtype=q_dtype, device=q.device)
        if k_out is None:
            ko = torch.empty((T, G * D), dtype=k_dtype or k.dtype, device=q.device)
            dst, sko, sl, nv = ko, G * D, None, 0
        else:
            nv = v.shape[1] if v is not None else 0
            assert k_out.shape[-1] >= G * D + nv and k_out.stride(-1) == 1 and slots is not None
            assert v_mix is None or (v is not None and v_mix.shape == v.shape and v_mix.dtype == v.dtype)
            ko, dst, sko, sl = None, k_out, k_out.shape[-1], slots
        N.mcall("mx_rope_heads", N.ptr(_rows(q)), q.stride(0), H, N.ptr(_rows(k)), k.stride(0), G, _dt(q), D, rot,
                1 if half else 0, N.ptr(freq), float(mscale), N.ptr(pos), 1 if norm else 0, float(norm_eps or 0.0),
                float(q_scale), float(k_scale), N.ptr(qo), _dt(qo), N.ptr(dst), sko, _dt(dst), N.ptr(sl),
                N.ptr(_rows(v)) if v is not None else None, v.stride(0) if v is not None else 0, nv,
                N.ptr(_rows(v_mix)) if v_mix is not None else None, v_mix.stride(0) if v_mix is not None else 0,
                float(v_lam), T, N.stream())
        return qo, ko
    ang = pos.float()[:, None] * freq.float()[None, :] if rot else None

    def prep(x, nh, sc):
        x = _rotate_heads(x.float().reshape(T, nh, D), ang, rot, half, mscale)
        if norm:
            x = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + norm_eps)
        return (x * sc).reshape(T, nh * D)

    qo = prep(q, H, q_scale).to(q_dtype)
    kk = prep(k, G, k_scale)
    if k_out is None:
        return qo, kk.to(k_dtype or k.dtype)
    vv = v.float() if v is not None else None
    if v_mix is not None:
        vv = (1.0 - v_lam) * vv + v_lam * v_mix.float()
    rows = torch.cat([kk] + ([vv] if vv is not None else []), 1).to(k_out.dtype)
    ok = slots >= 0
    k_out.view(-1, k_out.shape[-1])[slots[ok].long(), :rows.shape[1]] = rows[ok]
    return qo, None


# ----------------------------------------------------------------------------------------------
# matrix-state recurrence with one fixed decay per head
# ----------------------------------------------------------------------------------------------
def decay_scan(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, decay: torch.Tensor, state: torch.Tensor,
               cu: torch.Tensor, slot: torch.Tensor, pos: torch.Tensor, heads: int, dim: int, vdim: int,
               act: str = "none", out_scale: float = 1.0, max_len: int = 0) -> torch.Tensor:
    """Token-by-token f32 recurrence over a [dim, vdim] state per head with a constant decay per head:
    S <- decay[h] S + act(k) act(v)^T, o = S^T act(q) * out_scale.  ``q``, ``k`` [T, H*dim] (one storage
    type) and ``v`` [T, H*vdim] (possibly another) are column slices; ``act``: none | silu, applied to
    all three; ``decay`` f32 [H]; ``state`` f32 [slots, H, dim, vdim], read unless the segment starts at
    position 0, then replaced.  Returns o f32 [T, H*vdim]."""
    T = q.shape[0]
    H, D, P = heads, dim, vdim
    S = cu.numel() - 1
    assert q.dtype == k.dtype and q.shape[1] == H * D and k.shape[1] == H * D and v.shape[1] == H * P
    assert decay.dtype == torch.float32 and decay.numel() == H and act in ("none", "silu")
    if N.use_native(q):
        out = torch.empty((T, H * P), dtype=torch.float32, device=q.device)
        N.mcall("mx_decay_scan", N.ptr(_rows(q)), q.stride(0), N.ptr(_rows(k)), k.stride(0), _dt(q), N.ptr(_rows(v)),
                v.stride(0), _dt(v), ACTS[act], N.ptr(decay), float(out_scale), N.ptr(state), N.ptr(cu), N.ptr(slot),
                N.ptr(pos), N.ptr(out), S, T, int(max_len), H, D, P, N.stream())
        return out
    out = torch.zeros((T, H * P), dtype=torch.float32)
    cul, sll, pl = cu.tolist(), slot.tolist(), pos.tolist()
    g = decay.float()[:, None, None]
    for s in range(S):
        r0, r1 = cul[s], cul[s + 1]
        if sll[s] < 0 or r1 <= r0:
            continue
        n = r1 - r0
        qq = _act(q[r0:r1].float(), act).view(n, H, D)
        kk = _act(k[r0:r1].float(), act).view(n, H, D)
        vv = _act(v[r0:r1].float(), act).view(n, H, P)
        St = torch.zeros((H, D, P)) if pl[r0] == 0 else state[sll[s]].clone()
        for t in range(n):
            St = g * St + kk[t][:, :, None] * vv[t][:, None, :]
            out[r0 + t] = (torch.einsum("hdp,hd->hp", St, qq[t]) * out_scale).reshape(-1)
        state[sll[s]] = St
    return out
