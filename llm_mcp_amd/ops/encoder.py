"""The layers of an embedding encoder in one native call (csrc/kernels/encoder.hip).

``batch`` lays a batch of packed sequences out (positions, attention tiles), ``layers``
runs all layers.  The models keep their own
loop over single ops for the CPU and for shapes and switches this one does not take.
"""
from __future__ import annotations

import os
from dataclasses import dataclass

import numpy as np
import torch

PAGE = 32                      # of the models' own loops
QUERIES = 128                  # EA_Q in csrc/kernels/encattn.hip


@dataclass
class Batch:
    """Index arrays of packed sequences (device, int32)."""
    positions: torch.Tensor    # [T]
    tiles: torch.Tensor        # [2 * tiles] (sequence, first query), longest sequences first
    first: torch.Tensor        # [S] row of a sequence's first token
    count: torch.Tensor        # [S + 1] 0, 1, 2, ...
    longest: int


def batch(lens, device) -> Batch:
    """One upload for all arrays."""
    ln = np.asarray(lens, dtype=np.int32)
    S, T = len(ln), int(ln.sum())
    order = np.argsort(-ln, kind="stable").astype(np.int32)
    nt = -(-ln[order] // QUERIES)
    row0, tile0 = np.cumsum(ln) - ln, np.cumsum(nt) - nt
    NT = int(nt.sum())
    sizes = (T, 2 * NT, S, S + 1)
    at = np.concatenate([[0], np.cumsum([-(-n // 4) * 4 for n in sizes])])
    cuda = device.type == "cuda"
    host = torch.empty(int(at[-1]), dtype=torch.int32, pin_memory=cuda)
    h = host.numpy()
    pos, tiles, first, count = (h[a:a + n] for a, n in zip(at, sizes))
    pos[:] = np.arange(T, dtype=np.int32)
    pos -= np.repeat(row0, ln)
    tiles[0::2] = np.repeat(order, nt)
    tiles[1::2] = (np.arange(NT, dtype=np.int32) - np.repeat(tile0, nt)) * QUERIES
    first[:], count[:] = row0, np.arange(S + 1)
    dev = host.to(device, non_blocking=True) if cuda else host
    return Batch(*(dev[a:a + n] for a, n in zip(at.tolist(), sizes)), int(ln.max(initial=0)))


def layers_ok(layers: list, names: tuple, d: int, I: int, H: int, D: int) -> bool:
    """Whether the native layers run these weights: whole 256-column tiles, bf16 rows
    as they are stored, no switch that asks for the library."""
    if (d % 256 or I % 256 or d > 2048 or d != H * D or D != 64
            or os.environ.get("LMX_ENCODER_LIBRARY", "0") == "1"):
        return False
    return all(t is not None and t.dtype is torch.bfloat16 and t.is_contiguous()
               for L in layers for t in (L.get(n) for n in names))


def embed_norm(ids: torch.Tensor, word: torch.Tensor, type_row: torch.Tensor, w, b, eps: float,
               pos: torch.Tensor | None = None, positions: torch.Tensor | None = None) -> torch.Tensor:
    """LayerNorm(word[ids] + type (+ pos[positions])), bf16 rows."""
    from . import _ptr, _stream, native
    out = torch.empty((ids.numel(), word.shape[1]), dtype=word.dtype, device=word.device)
    native().embed_layernorm(_ptr(out), _ptr(ids), _ptr(word), word.shape[0], _ptr(type_row), _ptr(pos),
                             _ptr(positions), _ptr(w), _ptr(b), ids.numel(), word.shape[1], float(eps),
                             _stream())
    return out


def layers(x: torch.Tensor, weights: list, names: tuple, b: Batch, cu: torch.Tensor, I: int, H: int,
           D: int, eps: float, scale: float, gelu: bool,
           cos_sin: torch.Tensor | None) -> torch.Tensor:
    """All layers over x [T, d], in place.  ``names``: a layer's tensors in the order of
    encoder.h (None: the model has none there)."""
    from . import PGEMM_CALLS, _chk, _ptr, _stream, native, pgemm_counters
    T, d = x.shape
    _chk(cos_sin is None or b.longest <= cos_sin.shape[0], "a sequence is longer than cos_sin")
    dev, n = x.device, native().enc_slab_floats(T, d, I)
    rows = torch.empty(T * (5 * d + I), dtype=x.dtype, device=dev)       # h, attn, qkv, g
    at = [0, T * d, 2 * T * d, 5 * T * d]
    h, attn, qkv, g = (_ptr(rows) + 2 * a for a in at)
    tail = native().enc_tail_floats(T, d, I, gelu)
    if torch.cuda.is_current_stream_capturing():
        tail = 0               # see ops.pgemm_tail
    slabs = torch.empty(n + tail, dtype=torch.float32, device=dev)
    cnt = pgemm_counters(dev) if tail else None
    ptrs = [0 if k is None else L[k].data_ptr() for L in weights for k in names]
    native().encoder_layers(
        ptrs, T, d, I, H, D, gelu, float(eps), float(scale), _ptr(x), h, qkv, attn, g, _ptr(slabs), n,
        _ptr(cos_sin), _ptr(cu), _ptr(b.tiles), b.tiles.numel() // 2,
        _ptr(slabs) + 4 * n if tail else 0, tail, _ptr(cnt), _stream())
    PGEMM_CALLS[0] += 4 * len(weights)
    return x


def attention(qkv: torch.Tensor, cu: torch.Tensor, b: Batch, H: int, scale: float,
              cos_sin: torch.Tensor | None = None, rescale_thr: float = 8.0) -> torch.Tensor:
    """K24 alone: bidirectional attention of the packed sequences in the rows of qkv
    [T, 3 H 64] (``rescale_thr``: how far weights may exceed 1 before the maximum is raised, log2)."""
    from . import _chk, _ptr, _stream, native
    T, D = qkv.shape[0], qkv.shape[1] // (3 * H)
    _chk(qkv.dtype is torch.bfloat16 and qkv.stride(1) == 1, "qkv rows")
    _chk(cos_sin is None or (cos_sin.dtype is torch.float32 and cos_sin.is_contiguous()
                             and cos_sin.shape[0] >= b.longest), "cos_sin")
    out = torch.empty((T, H * D), dtype=qkv.dtype, device=qkv.device)
    native().enc_attention(_ptr(qkv), qkv.stride(0), H, D, _ptr(cu), _ptr(b.tiles), b.tiles.numel() // 2,
                           _ptr(cos_sin), _ptr(out), H * D, float(scale), float(rescale_thr), _stream())
    return out
