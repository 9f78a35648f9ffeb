"""The layers of an embedding encoder in one native call (csrc/kernels/encoder.hip).

``encode`` is a whole forward up to the pooling: ``batch`` lays the packed sequences out
(positions, attention tiles), ``embed_norm`` makes their rows, ``layers`` runs all layers.  The
kernels get addresses and the configuration's sizes, so everything they read is checked
first (``layers_ok``, ``embed_ok``); operands of several devices are refused.  The models keep
their own loop over single ops for the CPU and for operands and switches this one does not take.
"""
from __future__ import annotations

import functools
import itertools
import operator
import os
from dataclasses import dataclass

import numpy as np
import torch

PAGE = 32                      # of the models' own loops
QUERIES = 128                  # EA_Q in csrc/kernels/encattn.hip
LAYER_CALLS = [0]              # host-side count of layers run natively (enc_plan: on which kernels)


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
    at = [0, *itertools.accumulate(-(-n // 4) * 4 for n in sizes)]
    cuda = device.type == "cuda"
    host = torch.empty(at[-1], dtype=torch.int32, pin_memory=cuda)
    h = host.numpy()
    pos, tiles, first, count = (h[a:a + n] for a, n in zip(at, sizes))
    pos[:] = np.arange(T, dtype=np.int32)
    pos -= np.repeat(row0, ln)
    tiles[0::2] = np.repeat(order, nt)
    tiles[1::2] = (np.arange(NT, dtype=np.int32) - np.repeat(tile0, nt)) * QUERIES
    first[:], count[:] = row0, np.arange(S + 1)
    dev = host.to(device, non_blocking=True) if cuda else host
    return Batch(*(dev[a:a + n] for a, n in zip(at, sizes)), int(ln.max(initial=0)))


@functools.lru_cache(maxsize=64)
def _shapes(d: int, I: int, gelu: bool) -> tuple:
    """Shapes of a layer's tensors in the order of encoder.h."""
    v, w1 = (d,), I if gelu else 2 * I
    return tuple(torch.Size(s) for s in ((3 * d, d), (3 * d,), (d, d), v, v, v, (w1, d), (w1,), (d, I),
                                         v, v, v))


def sizes_ok(d: int, I: int, H: int, D: int, gelu: bool) -> bool:
    """Whether the native layers run an encoder of these sizes: whole 256-column tiles, a bias
    that K13 holds, no switch that asks for the library."""
    from . import PGEMM_MAX_BIAS
    return (d % 256 == 0 and I % 256 == 0 and d <= 2048 and d == H * D and D == 64
            and not (gelu and I > PGEMM_MAX_BIAS) and os.environ.get("LMX_ENCODER_LIBRARY", "0") != "1")


def _one_device(device: int, *tensors) -> None:
    """All are on the device of this index (-1: host)."""
    for t in tensors:
        if t is not None and t.get_device() != device:
            raise ValueError(f"an encoder operand on {t.device}, its rows on device {device}")


def weights_on(ids: torch.Tensor, cu: torch.Tensor, w: dict, names: tuple,
               cos_sin: torch.Tensor | None = None) -> None:
    """Everything that a forward reads (``names`` of a layer) is on the rows' device.  Before the
    models' own loop, whose kernels get addresses too."""
    device = ids.get_device()
    _one_device(device, cu, cos_sin, *(w.get(n) for n in ("word", "type", "emb_ln_w", "emb_ln_b")),
                w.get("pos") if cos_sin is None else None)
    for L in w["layers"]:
        _one_device(device, *(L.get(n) for n in names))


def layers_ok(layers: list, names: tuple, d: int, I: int, gelu: bool, device: int = -1) -> list | None:
    """Addresses of the layers' weights, ``names`` of them a layer (None: the model has none
    there), if all are bf16 tensors of the configuration's shapes as they are stored, on 16
    bytes.  Else None: the models' own loop takes or refuses them.  ``device``: _one_device's."""
    want, bf16, out = list(zip(names, _shapes(d, I, gelu))), torch.bfloat16, []
    for L in layers:
        for n, shape in want:
            if n is None:
                out.append(0)
                continue
            t = L.get(n)
            if t is None or t.dtype is not bf16 or t.shape != shape or not t.is_contiguous():
                return None
            if t.get_device() != device:
                _one_device(device, t)
            out.append(t.data_ptr())
    return None if functools.reduce(operator.or_, out, 0) & 15 else out


def _rows_ok(t: torch.Tensor, cols: int, dims: int = 2) -> bool:
    return (t.dtype is torch.bfloat16 and t.dim() == dims and t.shape[-1] == cols and t.is_contiguous()
            and t.data_ptr() % 16 == 0)


def _rotary_ok(t: torch.Tensor, D: int) -> bool:
    return (t.dtype is torch.float32 and t.dim() == 2 and t.shape[1] == D and t.is_contiguous()
            and t.data_ptr() % 16 == 0)


def _index_ok(t: torch.Tensor, n: int) -> bool:
    return t.dtype is torch.int32 and t.dim() == 1 and t.numel() == n and t.is_contiguous()


def embed_ok(ids: torch.Tensor, word: torch.Tensor, type_row: torch.Tensor, w, b,
             pos: torch.Tensor | None = None, positions: torch.Tensor | None = None) -> bool:
    """Whether ``embed_norm`` reads these, all on one device (``_one_device``): int32 indices,
    contiguous bf16 tables and vectors of one width on 16 bytes."""
    d = word.shape[-1]
    return (_index_ok(ids, ids.numel()) and _rows_ok(word, d) and d % 8 == 0 and d <= 2048
            and _rows_ok(type_row, d) and type_row.shape[0] > 0 and _rows_ok(w, d, 1) and _rows_ok(b, d, 1)
            and (pos is None or _rows_ok(pos, d))
            and (positions is None or _index_ok(positions, ids.numel())))


def embed_norm(ids: torch.Tensor, word: torch.Tensor, type_row: torch.Tensor, w, b, eps: float,
               pos: torch.Tensor | None = None, positions: torch.Tensor | None = None) -> torch.Tensor:
    """LayerNorm(word[ids] + type (+ pos[positions])), bf16 rows.  ``positions`` are the caller's
    to keep below pos's rows."""
    from . import _chk
    _one_device(ids.get_device(), word, type_row, w, b, pos, positions)
    _chk(embed_ok(ids, word, type_row, w, b, pos, positions)
         and (pos is None or positions is not None), "embed_norm operands")
    return _embed_norm(ids, word, type_row, w, b, eps, pos, positions)


def _embed_norm(ids, word, type_row, w, b, eps, pos, positions) -> torch.Tensor:
    from . import _ptr, _stream, native
    out = torch.empty((ids.numel(), word.shape[1]), dtype=word.dtype, device=word.device)
    native().embed_layernorm(_ptr(out), _ptr(ids), _ptr(word), word.shape[0], _ptr(type_row), _ptr(pos),
                             _ptr(positions), _ptr(w), _ptr(b), ids.numel(), word.shape[1], float(eps),
                             _stream())
    return out


def encode(ids: torch.Tensor, cu: torch.Tensor, lens: list, w: dict, names: tuple, cfg, scale: float,
           gelu: bool, cos_sin: torch.Tensor | None = None) -> tuple | None:
    """(rows [T, d] after all layers, their ``Batch``) of packed sequences, or None where the
    native layers do not take these operands (the models' own loop takes or refuses them).
    ``cos_sin``: rotary tables; without them w["pos"] holds a row for every position."""
    from . import _chk
    d, I, H, D = cfg.hidden_size, cfg.intermediate_size, cfg.num_heads, cfg.head_dim
    word, pos = w["word"], None if cos_sin is not None else w["pos"]
    device = ids.get_device()
    _one_device(device, cu, word, w["type"], w["emb_ln_w"], w["emb_ln_b"], pos, cos_sin)
    if not (sizes_ok(d, I, H, D, gelu) and word.shape[-1] == d and sum(lens) == ids.numel() > 0
            and _index_ok(cu, len(lens) + 1)
            and embed_ok(ids, word, w["type"], w["emb_ln_w"], w["emb_ln_b"], pos)
            and (cos_sin is None or _rotary_ok(cos_sin, D))):
        return None
    b = batch(lens, ids.device)
    _chk(b.longest <= (pos if cos_sin is None else cos_sin).shape[0],
         "a sequence is longer than the position table")
    x = _embed_norm(ids, word, w["type"], w["emb_ln_w"], w["emb_ln_b"], cfg.ln_eps, pos,
                    b.positions if pos is not None else None)
    # here, while the upload and the first norm run (50 us for 12 layers)
    ptrs = layers_ok(w["layers"], names, d, I, gelu, device)
    return (layers(x, ptrs, b, cu, I, H, D, cfg.ln_eps, scale, gelu, cos_sin), b) if ptrs else None


def layers(x: torch.Tensor, ptrs: list, b: Batch, cu: torch.Tensor, I: int, H: int, D: int, eps: float,
           scale: float, gelu: bool, cos_sin: torch.Tensor | None) -> torch.Tensor:
    """All layers over x [T, d], in place.  ``ptrs``: ``layers_ok``'s."""
    from . import _ptr, _stream, native, pgemm_tail_memory
    T, d = x.shape
    dev, n = x.device, native().enc_slab_floats(T, d, I)
    rows = torch.empty(T * (5 * d + I), dtype=x.dtype, device=dev)       # h, attn, qkv, g
    at = [0, T * d, 2 * T * d, 5 * T * d]
    h, attn, qkv, g = (_ptr(rows) + 2 * a for a in at)
    slabs = torch.empty(n, dtype=torch.float32, device=dev)
    tail, cnt = pgemm_tail_memory(dev, native().enc_tail_floats(T, d, I, gelu))
    native().encoder_layers(
        ptrs, T, d, I, H, D, gelu, float(eps), float(scale), _ptr(x), h, qkv, attn, g, _ptr(slabs), n,
        _ptr(cos_sin), _ptr(cu), _ptr(b.tiles), b.tiles.numel() // 2,
        _ptr(tail), 0 if tail is None else tail.numel(), _ptr(cnt), _stream())
    LAYER_CALLS[0] += len(ptrs) // 12
    return x


def attention(qkv: torch.Tensor, cu: torch.Tensor, b: Batch, H: int, scale: float,
              cos_sin: torch.Tensor | None = None, rescale_thr: float = 8.0) -> torch.Tensor:
    """K24 alone: bidirectional attention of the packed sequences in the rows of qkv
    [T, 3 H 64] (``rescale_thr``: how far weights may exceed 1 before the maximum is raised, log2)."""
    from . import _chk, _ptr, _stream, native
    T, D = qkv.shape[0], qkv.shape[1] // (3 * H)
    _chk(qkv.dtype is torch.bfloat16 and qkv.stride(1) == 1, "qkv rows")
    _chk(cos_sin is None or (_rotary_ok(cos_sin, D) and cos_sin.shape[0] >= b.longest), "cos_sin")
    out = torch.empty((T, H * D), dtype=qkv.dtype, device=qkv.device)
    native().enc_attention(_ptr(qkv), qkv.stride(0), H, D, _ptr(cu), _ptr(b.tiles), b.tiles.numel() // 2,
                           _ptr(cos_sin), _ptr(out), H * D, float(scale), float(rescale_thr), _stream())
    return out
