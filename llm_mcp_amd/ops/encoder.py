"""The layers of an embedding encoder in one native call (csrc/kernels/encoder.hip).

``batch`` lays a batch of packed sequences out for the paged attention (page slots,
positions, attention tiles), ``layers`` runs all layers.  The models keep their own
loop over single ops for the CPU and for shapes and switches this one does not take.
"""
from __future__ import annotations

import os
from dataclasses import dataclass

import numpy as np
import torch

PAGE = 32


@dataclass
class Batch:
    """Index arrays of packed sequences (device, int32)."""
    slots: torch.Tensor        # [T] place of a token in the scratch pages
    positions: torch.Tensor    # [T]
    tiles: torch.Tensor        # [2 * tiles] (sequence, first query)
    first: torch.Tensor        # [S] row of a sequence's first token
    ctx: torch.Tensor          # [S] lengths
    count: torch.Tensor        # [S + 1] 0, 1, 2, ...
    tables: torch.Tensor       # [S, most pages]
    pages: int


def batch(lens, q_per_tile: int, device) -> Batch:
    """Every sequence in whole pages of its own, one upload for all arrays."""
    ln = np.asarray(lens, dtype=np.int32)
    S, T = len(ln), int(ln.sum())
    pages, nt = np.maximum(1, -(-ln // PAGE)), -(-ln // q_per_tile)
    page0, row0, tile0 = (np.cumsum(a) - a for a in (pages, ln, nt))
    NB, NT, most = int(pages.sum()), int(nt.sum()), int(pages.max())
    sizes = (T, T, 2 * NT, S, S, S + 1, S * most)
    at = np.concatenate([[0], np.cumsum([-(-n // 4) * 4 for n in sizes])])
    cuda = device.type == "cuda"
    host = torch.empty(int(at[-1]), dtype=torch.int32, pin_memory=cuda)
    h = host.numpy()
    slots, pos, tiles, first, ctx, count, tables = (h[a:a + n] for a, n in zip(at, sizes))
    pos[:] = np.arange(T, dtype=np.int32)
    pos -= np.repeat(row0, ln)
    np.add(np.repeat(page0 * PAGE, ln), pos, out=slots)
    seq = np.repeat(np.arange(S, dtype=np.int32), nt)
    tiles[0::2] = seq
    tiles[1::2] = (np.arange(NT, dtype=np.int32) - tile0[seq]) * q_per_tile
    first[:], ctx[:], count[:] = row0, ln, np.arange(S + 1)
    # columns past a sequence's pages are never read
    np.minimum(page0[:, None] + np.arange(most, dtype=np.int32), NB - 1,
               out=tables.reshape(S, most), casting="unsafe")
    dev = host.to(device, non_blocking=True) if cuda else host
    d = [dev[a:a + n] for a, n in zip(at.tolist(), sizes)]
    return Batch(*d[:6], d[6].view(S, most), NB)


def layers_ok(layers: list, names: tuple, d: int, I: int, H: int, D: int) -> bool:
    """Whether the native layers run these weights: whole 256-column tiles, bf16 rows
    as they are stored, no switch that asks for the library."""
    if (d % 256 or I % 256 or d > 2048 or d != H * D or D not in (64, 128)
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
           D: int, eps: float, scale: float, q_per_tile: int, gelu: bool,
           cos_sin: torch.Tensor | None) -> torch.Tensor:
    """All layers over x [T, d], in place.  ``names``: a layer's tensors in the order of
    encoder.h (None: the model has none there)."""
    from . import PGEMM_CALLS, _ptr, _stream, native, pgemm_counters
    T, d = x.shape
    dev, n = x.device, native().enc_slab_floats(T, d, I)
    rows = torch.empty(T * (5 * d + I), dtype=x.dtype, device=dev)       # h, attn, qkv, g
    at = [0, T * d, 2 * T * d, 5 * T * d]
    h, attn, qkv, g = (_ptr(rows) + 2 * a for a in at)
    tail = native().enc_tail_floats(T, d, I, gelu)
    if torch.cuda.is_current_stream_capturing():
        tail = 0               # see ops.pgemm_tail
    slabs = torch.empty(n + tail, dtype=torch.float32, device=dev)
    cnt = pgemm_counters(dev) if tail else None
    # masked keys weigh 0 times V, which must be finite
    kv = torch.zeros(2 * b.pages * H * PAGE * D, dtype=x.dtype, device=dev)
    ptrs = [0 if k is None else L[k].data_ptr() for L in weights for k in names]
    native().encoder_layers(
        ptrs, T, d, I, H, D, PAGE, gelu, float(eps), float(scale), _ptr(x), h, qkv, attn, g,
        _ptr(slabs), n, _ptr(kv), _ptr(kv) + kv.numel(), _ptr(b.slots), _ptr(b.positions),
        _ptr(cos_sin), _ptr(b.tables), b.tables.stride(0), _ptr(cu), _ptr(b.ctx), _ptr(b.tiles),
        b.tiles.numel() // 2, q_per_tile, _ptr(slabs) + 4 * n if tail else 0, tail, _ptr(cnt),
        _stream())
    PGEMM_CALLS[0] += 4 * len(weights)
    return x
