"""BERT / bge-base-en encoder on the GPU (replaces OpenAIEmbeddings, qdrant_tool.py:28).

Post-LN BERT: embeddings (word + position + type) -> LayerNorm -> 12 x [fused QKV GEMM (+bias)
-> bidirectional attention -> O GEMM -> add+LayerNorm -> GELU MLP -> add+LayerNorm] -> CLS
pooling -> L2 normalise.  Queries are packed varlen (no padding FLOPs); attention reads the packed QKV
rows as they are (``csrc/kernels/encoder.hip``).
"""
from __future__ import annotations

import ctypes
import math
import os
from typing import Dict, Optional, Sequence, Tuple

import numpy as np
import torch
import torch.nn.functional as F

from .. import ops
from ..ops import _native as N
from ..ops.gemm import BGE_SMALL_MAX_M, SMALL_MAX_MADS, linear_bias
from .common import random_tensor
from .configs import ModelConfig


# a layer's weights, in the order of penny_encoder_layers
LAYER = ("qkv", "qkv_b", "o", "o_b", "ln1_g", "ln1_b", "fc1", "fc1_b", "fc2", "fc2_b", "ln2_g", "ln2_b")


EMBED_ARGS = 960             # ints that travel with penny_encoder_embed_host's launch


class BertEncoder:
    def __init__(self, cfg: ModelConfig, device="cuda", dtype=torch.bfloat16):
        self.cfg = cfg
        self.device = torch.device(device)
        self.dtype = dtype
        self.H, self.nh, self.D = cfg.hidden_size, cfg.num_heads, cfg.head_dim
        self.w: Dict[str, torch.Tensor] = {}
        self.layer_names = [f"layers.{i}.{n}" for i in range(cfg.num_layers) for n in LAYER]
        shapes = self.shapes()
        self.layer_shapes = [shapes[n] for n in self.layer_names]

    def shapes(self) -> Dict[str, tuple]:
        c = self.cfg
        H, F_ = c.hidden_size, c.intermediate_size
        s = {"word_emb": (c.vocab_size, H), "pos_emb": (c.max_position, H), "type_emb": (c.type_vocab_size, H),
             "emb_ln_g": (H,), "emb_ln_b": (H,)}
        for i in range(c.num_layers):
            p = f"layers.{i}."
            s.update({p + "qkv": (3 * H, H), p + "qkv_b": (3 * H,), p + "o": (H, H), p + "o_b": (H,),
                      p + "ln1_g": (H,), p + "ln1_b": (H,), p + "fc1": (F_, H), p + "fc1_b": (F_,),
                      p + "fc2": (H, F_), p + "fc2_b": (H,), p + "ln2_g": (H,), p + "ln2_b": (H,)})
        return s

    @classmethod
    def build(cls, cfg: ModelConfig, device="cuda", weights: Optional[str] = None, seed: int = 0,
              dtype=torch.bfloat16) -> "BertEncoder":
        m = cls(cfg, device, dtype)
        if weights:
            from .weights import hf_bert_to_internal, read_safetensors
            m.load_state(hf_bert_to_internal(read_safetensors(weights), cfg.num_layers))
        else:
            for name, shape in m.shapes().items():
                kind = "ones" if name.endswith("_g") else ("zeros" if name.endswith("_b") else "normal")
                m.w[name] = random_tensor("bert." + name, shape, seed, m.device, dtype, kind=kind)
        return m

    def load_state(self, sd: Dict[str, torch.Tensor]) -> "BertEncoder":
        for k, v in sd.items():
            self.w[k] = v.to(self.device, self.dtype).contiguous()
        return self

    def _embed_rows(self) -> Optional[list]:
        """The embedding's five tensors where the native pass takes them."""
        rows = [self.w[n] for n in ("word_emb", "pos_emb", "type_emb", "emb_ln_g", "emb_ln_b")]
        return rows if N.use_native(rows[0]) and self.H in (256, 512, 768, 1024) and \
            all(t.dtype == torch.bfloat16 and t.is_contiguous() and t.shape[-1] == self.H for t in rows) else None

    def _embed(self, ids: torch.Tensor, pos: torch.Tensor) -> torch.Tensor:
        c, w, rows = self.cfg, self.w, self._embed_rows()
        if rows is not None:
            x = torch.empty((ids.numel(), self.H), dtype=torch.bfloat16, device=ids.device)
            word, position, kind, g, b = rows
            N.call("penny_encoder_embed", N.ptr(ids), N.ptr(pos), N.ptr(word), word.shape[0], N.ptr(position),
                   position.shape[0], N.ptr(kind), N.ptr(g), N.ptr(b), N.ptr(x), x.shape[0], self.H, float(c.norm_eps), N.stream())
            return x
        e_word = ops.embedding(ids, w["word_emb"])
        e_pos = ops.embedding(pos, w["pos_emb"])
        e_pos = (e_pos.float() + w["type_emb"][0].float()).to(self.dtype)
        return ops.layer_norm(e_word, w["emb_ln_g"], w["emb_ln_b"], c.norm_eps, residual=e_pos)

    def _small_batch(self, x: torch.Tensor, cu: torch.Tensor, longest: int) -> bool:
        """All layers of a batch of up to BGE_SMALL_MAX_M tokens (fewer in wide models), or of more where every projection is one round
        of blocks, in one native call (x in place); False: not a case for it."""
        T, F_ = x.shape[0], self.cfg.intermediate_size
        if not (N.use_native(x) and (T <= BGE_SMALL_MAX_M and T * self.H * max(F_, 3 * self.H) < SMALL_MAX_MADS or T <= 2048 and all(
                N.load().penny_bias_rows_plan(T, n, k) for n, k in ((3 * self.H, self.H), (self.H, self.H), (F_, self.H), (self.H, F_)))) and
                x.dtype == torch.bfloat16 and cu.numel() <= 65536 and self.H % 32 == 0 and F_ % 32 == 0 and
                os.environ.get("PENNY_PREFILL_GEMM", "1") == "1"):
            return False
        w = [self.w[n] for n in self.layer_names]
        if not all(t.dtype == torch.bfloat16 and t.is_contiguous() and t.device == x.device for t in w) or \
                [t.shape for t in w] != self.layer_shapes:
            return False
        table = (ctypes.c_void_p * len(w))(*[t.data_ptr() for t in w])
        lib = N.load()
        slices = lib.penny_encoder_slices(T, self.H, F_)
        scratch = torch.empty(T * (6 * self.H + F_ + (2 * slices * self.H if slices > 1 else 0)), dtype=torch.bfloat16, device=x.device)
        rc = lib.penny_encoder_layers(table, self.cfg.num_layers, N.ptr(x), N.ptr(scratch), N.ptr(cu), cu.numel() - 1, longest,
                                           T, self.H, self.nh, F_, float(self.cfg.norm_eps), 1.0 / math.sqrt(self.D), N.stream())
        if rc > 0:
            raise RuntimeError(f"penny_encoder_layers failed with hipError {rc}")
        return rc == 0                       # else a weight off the kernels' 16 bytes, and nothing was launched

    def _hidden(self, ids_list: Sequence[Sequence[int]]) -> Tuple[torch.Tensor, np.ndarray, torch.Tensor]:
        c, dev = self.cfg, self.device
        # packed varlen metadata, vectorised on the host (bulk ingest packs 100k+ tokens a call)
        lens = np.fromiter((len(x) for x in ids_list), np.int64, len(ids_list))
        T = int(lens.sum())
        cu = np.zeros(len(lens) + 1, np.int64)
        np.cumsum(lens, out=cu[1:])
        # token ids | positions | row bounds: one copy to the device
        meta = np.empty(2 * T + len(cu), np.int32)
        meta[:T] = np.fromiter((t for x in ids_list for t in x), np.int32, T)
        meta[T:2 * T] = np.arange(T, dtype=np.int64) - np.repeat(cu[:-1], lens)
        meta[2 * T:] = cu
        longest = int(lens.max())
        w, rows = self.w, self._embed_rows()
        # a recorded launch would hold this call's ids: a capture meets the copy
        if 0 < T and len(meta) <= EMBED_ARGS and rows is not None and not torch.cuda.is_current_stream_capturing():
            word, position, kind, g, b = rows
            x = torch.empty((T, self.H), dtype=torch.bfloat16, device=dev)
            cu_t = torch.empty(len(cu), dtype=torch.int32, device=dev)
            N.call("penny_encoder_embed_host", meta.ctypes.data, len(cu), N.ptr(word), word.shape[0], N.ptr(position), position.shape[0],
                   N.ptr(kind), N.ptr(g), N.ptr(b), N.ptr(x), T, self.H, float(c.norm_eps), N.ptr(cu_t), N.stream())
        else:
            ids_t, pos_t, cu_t = torch.from_numpy(meta).to(dev).split([T, T, len(cu)])
            x = self._embed(ids_t, pos_t)
        if self._small_batch(x, cu_t, longest):
            return x, cu, cu_t
        scale = 1.0 / math.sqrt(self.D)
        for i in range(c.num_layers):
            p = f"layers.{i}."
            qkv = linear_bias(x, w[p + "qkv"], w[p + "qkv_b"])
            a = ops.encoder_attention(qkv, cu_t, longest, self.nh, scale)
            o = linear_bias(a, w[p + "o"], w[p + "o_b"])
            x = ops.layer_norm(o, w[p + "ln1_g"], w[p + "ln1_b"], c.norm_eps, residual=x)
            h = linear_bias(x, w[p + "fc1"], w[p + "fc1_b"], gelu=True)      # bias + GELU fused
            y = linear_bias(h, w[p + "fc2"], w[p + "fc2_b"])
            x = ops.layer_norm(y, w[p + "ln2_g"], w[p + "ln2_b"], c.norm_eps, residual=x)
        return x, cu, cu_t

    @torch.no_grad()
    def forward(self, ids_list: Sequence[Sequence[int]]) -> torch.Tensor:
        """-> final hidden states [T, H] of the packed batch, plus CLS row indices."""
        x, cu, _ = self._hidden(ids_list)
        return x, cu.tolist()

    @torch.no_grad()
    def encode(self, ids_list: Sequence[Sequence[int]]) -> torch.Tensor:
        """CLS pooling + L2 normalisation (bge convention) -> [n, H] f32."""
        x, cu, cu_t = self._hidden(ids_list)
        if N.use_native(x) and x.dtype == torch.bfloat16 and cu[-2] < x.shape[0]:
            out = torch.empty((len(cu) - 1, self.H), dtype=torch.float32, device=x.device)
            N.call("penny_encoder_pool", N.ptr(x), N.ptr(cu_t), len(cu) - 1, self.H, N.ptr(out), N.stream())
            return out
        cls = x[torch.tensor(cu[:-1].tolist(), device=x.device)]
        return F.normalize(cls.float(), dim=-1)
