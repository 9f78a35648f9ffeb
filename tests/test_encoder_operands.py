"""Which operands the encoders' native layers take (ops.encoder): the kernels get addresses and the
configuration's sizes, so all others go to the models' own loop or are refused."""
import dataclasses
import types

import pytest
import torch

from llm_mcp_amd import ops
from llm_mcp_amd.models import bert, nomic_bert
from llm_mcp_amd.models import config as mc
from llm_mcp_amd.ops import encoder

D, I, V, P = 256, 512, 40, 20
LENS = [7, 1, 12]


def _zeros(*shape):
    return torch.zeros(shape, dtype=torch.bfloat16)


def _model(gelu):
    names = bert.NATIVE if gelu else nomic_bert.NATIVE
    shapes = encoder._shapes(D, I, gelu)
    return names, dict(word=_zeros(V, D), type=_zeros(2, D), pos=_zeros(P, D), emb_ln_w=_zeros(D),
                       emb_ln_b=_zeros(D),
                       layers=[{n: _zeros(*s) for n, s in zip(names, shapes) if n} for _ in range(2)])


def _ok(names, w, gelu):
    return encoder.layers_ok(w["layers"], names, D, I, gelu)


def _encode(names, w, gelu, ids=None, cu=None, lens=LENS, rows=P, cos_sin=None):
    cfg = types.SimpleNamespace(hidden_size=D, intermediate_size=I, num_heads=D // 64, head_dim=64,
                                ln_eps=1e-12)
    ids = torch.zeros(sum(LENS), dtype=torch.int32) if ids is None else ids
    cu = torch.tensor([0, 7, 8, 20], dtype=torch.int32) if cu is None else cu
    cos_sin = torch.zeros(rows, 64) if cos_sin is None else cos_sin
    return encoder.encode(ids, cu, lens, w, names, cfg, 0.125, gelu, None if gelu else cos_sin)


class _Reached(Exception):
    pass


@pytest.fixture
def reached(monkeypatch):
    """The kernels' place: says that all checks were passed."""
    def stop(*a):
        raise _Reached
    monkeypatch.setattr(encoder, "_embed_norm", lambda *a: None)
    monkeypatch.setattr(encoder, "layers", stop)


@pytest.mark.parametrize("gelu", [True, False])
def test_layers(gelu, reached):
    names, w = _model(gelu)
    addresses = _ok(names, w, gelu)
    assert addresses == [0 if n is None else L[n].data_ptr() for L in w["layers"] for n in names]
    with pytest.raises(_Reached):
        _encode(names, w, gelu)
    for n in filter(None, names):
        t = w["layers"][1][n]
        small = t[:-16].clone()                                    # fewer rows than the configuration says
        off = torch.zeros(t.numel() + 8, dtype=t.dtype)
        off = off[-off.data_ptr() // 2 % 8 + 1:][:t.numel()].view(t.shape)          # 2 bytes off a boundary
        bad = [None, small, t.float(), off]
        if t.dim() == 2:
            bad += [t[:, :-64].contiguous(), _zeros(t.shape[1], t.shape[0]).t(), t[:, :-64]]
        for b in bad:
            w["layers"][1][n] = b
            assert _ok(names, w, gelu) is None and _encode(names, w, gelu) is None, n
        w["layers"][1][n] = t


def test_bias_wider_than_k13_holds():
    assert encoder.sizes_ok(D, 14336, D // 64, 64, True) and not encoder.sizes_ok(D, 14592, D // 64, 64, True)
    assert encoder.sizes_ok(D, 14592, D // 64, 64, False)


@pytest.mark.parametrize("gelu", [True, False])
def test_embedding_and_indices(gelu, reached):
    names, w = _model(gelu)
    wide = torch.zeros(V, D + 8, dtype=torch.bfloat16)[:, :D]
    for n, bad in (("word", [w["word"].float(), wide, _zeros(V, D - 8)]), ("type", [w["type"].float()]),
                   ("emb_ln_w", [w["emb_ln_w"].float(), _zeros(D - 8)]), ("emb_ln_b", [_zeros(D + 8)]),
                   ("pos", [w["pos"].float(), wide])):
        if n == "pos" and not gelu:
            continue
        keep = w[n]
        for b in bad:
            w[n] = b
            assert _encode(names, w, gelu) is None, n
        w[n] = keep
    ids, cu = torch.zeros(sum(LENS), dtype=torch.int32), torch.tensor([0, 7, 8, 20], dtype=torch.int32)
    for kw in (dict(ids=ids.long()), dict(ids=ids[:-1]), dict(ids=torch.zeros(40, dtype=torch.int32)[::2]),
               dict(cu=cu.long()), dict(cu=cu[:-1]), dict(lens=[7, 1, 13]), dict(ids=ids[:0], cu=cu[:1], lens=[])):
        assert _encode(names, w, gelu, **kw) is None, kw


@pytest.mark.parametrize("gelu", [True, False])
def test_positions_within_their_table(gelu, reached):
    """A sequence longer than the positions' table is refused, not read past the table's end."""
    names, w = _model(gelu)
    w["pos"] = _zeros(11, D)
    with pytest.raises(ValueError):
        _encode(names, w, gelu, rows=11)
    w["pos"] = _zeros(12, D)
    with pytest.raises(_Reached):
        _encode(names, w, gelu, rows=12)


def test_rotary_table(reached):
    """fp32 rows of a head on 16 bytes: others go to the models' own loop, which takes an address
    off 16 bytes and whose rotation refuses the rest."""
    names, w = _model(False)
    t = torch.zeros(P, 64)
    off = torch.zeros(P * 64 + 4)
    off = off[-off.data_ptr() // 4 % 4 + 1:][:P * 64].view(P, 64)
    for bad in (t.bfloat16(), t[:, :32].contiguous(), torch.zeros(P, 128)[:, :64], t.flatten(), off):
        assert _encode(names, w, False, cos_sin=bad) is None
    with pytest.raises(_Reached):
        _encode(names, w, False, cos_sin=t)


class _Elsewhere(torch.Tensor):
    """A host tensor that says it is on a device."""
    def get_device(self):
        return 0


@pytest.mark.parametrize("gelu", [True, False])
def test_operands_of_several_devices(gelu, reached):
    """Refused, and not left to the models' own loop, whose kernels get addresses too."""
    names, w = _model(gelu)
    for n in ["word", "type", "emb_ln_w", "emb_ln_b"] + ["pos"] * gelu:
        with pytest.raises(ValueError):
            _encode(names, {**w, n: w[n].as_subclass(_Elsewhere)}, gelu)
    cu, ids = torch.tensor([0, 7, 8, 20], dtype=torch.int32), torch.zeros(5, dtype=torch.int32)
    for kw in ([dict(cu=cu.as_subclass(_Elsewhere))]
               + [dict(cos_sin=torch.zeros(P, 64).as_subclass(_Elsewhere))] * (not gelu)):
        with pytest.raises(ValueError):
            _encode(names, w, gelu, **kw)
    with pytest.raises(ValueError):
        encoder.embed_norm(ids, w["word"], w["type"].as_subclass(_Elsewhere), w["emb_ln_w"], w["emb_ln_b"], 1e-12)
    for n in filter(None, names):
        t = w["layers"][1][n]
        w["layers"][1][n] = t.as_subclass(_Elsewhere)
        with pytest.raises(ValueError):
            _encode(names, w, gelu)
        w["layers"][1][n] = t
    with pytest.raises(ValueError):
        encoder.layers_ok(w["layers"], names, D, I, gelu, 0)       # all of them on the host, the rows not


@pytest.mark.parametrize("gelu", [True, False])
def test_weights_on(gelu):
    """The check before the models' own loop: every tensor that it reads, and no other."""
    names, w = _model(gelu)
    ids, cu, cos_sin = torch.zeros(20, dtype=torch.int32), torch.tensor([0, 20], dtype=torch.int32), _zeros(P, 64)
    encoder.weights_on(ids, cu, w, names)
    away = lambda t: t.as_subclass(_Elsewhere)
    layer = lambda n, t: {**w, "layers": [w["layers"][0], {**w["layers"][1], n: t}]}
    encoder.weights_on(ids, cu, {**layer("other", away(cu)), "pos": away(cu), "note": "text"}, names, cos_sin)
    for args in ([(ids, away(cu), w, names, cos_sin), (ids, cu, w, names, away(cos_sin)), (away(ids), cu, w, names)]
                 + [(ids, cu, {**w, n: away(w[n])}, names) for n in w if n != "layers"]
                 + [(ids, cu, layer(n, away(t)), names) for n, t in w["layers"][1].items()]):
        with pytest.raises(ValueError):
            encoder.weights_on(*args)


@pytest.mark.gpu
@pytest.mark.parametrize("heads", [4, 2])
@pytest.mark.parametrize("model", ["tiny-bert", "tiny-nomic"])
def test_models_refuse_operands_of_several_devices(model, heads):
    """A weight left on the host, anywhere in the model: no kernel gets its address, on the native
    layers (heads of 64) and in the models' own loop."""
    cfg = dataclasses.replace(mc.resolve(model), num_heads=heads, head_dim=D // heads)
    gelu = cfg.family == "bert"
    m = (bert.BertModel if gelu else nomic_bert.NomicBertModel)(cfg, "cuda", seed=1)
    ids, cu = (torch.tensor(a, dtype=torch.int32) for a in (list(range(20)), [0, 7, 8, 20]))
    run = lambda c, i=ids.cuda(): m.forward(i, c, LENS)
    names = bert.NATIVE if gelu else nomic_bert.NATIVE
    for where, n in ([(m.w, n) for n in ("word", "type", "emb_ln_w", "emb_ln_b")] + [(m.w, "pos")] * gelu
                     + [(m.w["layers"][-1], n) for n in names if n]):
        keep = where[n]
        where[n] = keep.cpu()
        with pytest.raises(ValueError):
            run(cu.cuda())
        where[n] = keep
    for args in ((cu,), (cu.cuda(), ids), (cu, ids)):
        with pytest.raises(ValueError):
            run(*args)
    assert bool(run(cu.cuda()).isfinite().all())


def test_layer_norm_operands():
    """What the models' own loop passes to its LayerNorm by address."""
    x, v, r = _zeros(5, D), _zeros(D), _zeros(7, D)
    assert ops.layer_norm_ok(x, v, v) and ops.layer_norm_ok(x, v[None], v, r) and ops.layer_norm_ok(x, v, v, r[:5])
    for args in ((x.float(), v, v), (x, v.float(), v), (x, v, v.float()), (x, v[:-8], v), (x, v, _zeros(D + 8)),
                 (x, _zeros(2 * D)[::2], v), (x, v, v, x.float()), (x, v, v, x[:4]), (x, v, v, _zeros(D, 5).t()),
                 (x, v, v, _zeros(5, 2 * D)[:, :D]), (x, v, v, _zeros(10, D // 2)), (_zeros(D, 5).t(), v, v),
                 (x, v.as_subclass(_Elsewhere), v), (x, v, v.as_subclass(_Elsewhere)),
                 (x, v, v, r.as_subclass(_Elsewhere))):
        assert not ops.layer_norm_ok(*args)


@pytest.mark.gpu
@pytest.mark.parametrize("heads", [4, 2])
@pytest.mark.parametrize("model", ["tiny-bert", "tiny-nomic"])
def test_models_refuse_other_norm_weights(model, heads):
    cfg = dataclasses.replace(mc.resolve(model), num_heads=heads, head_dim=D // heads)
    m = (bert.BertModel if cfg.family == "bert" else nomic_bert.NomicBertModel)(cfg, "cuda", seed=1)
    ids, cu = (torch.tensor(a, dtype=torch.int32).cuda() for a in (list(range(20)), [0, 7, 8, 20]))
    for where, n in ((m.w, "emb_ln_w"), (m.w["layers"][0], "ln1_b"), (m.w["layers"][-1], "ln2_w")):
        keep = where[n]
        for bad in (keep.float(), keep[:-8].clone()):
            where[n] = bad
            with pytest.raises(ValueError):
                m.forward(ids, cu, LENS)
        where[n] = keep


@pytest.mark.gpu
@pytest.mark.parametrize("heads", [4, 2])
@pytest.mark.parametrize("model", ["tiny-bert", "tiny-nomic"])
def test_strided_indices(model, heads):
    """Every second element of an index array: the vectors of the loop on a contiguous copy."""
    cfg = dataclasses.replace(mc.resolve(model), num_heads=heads, head_dim=D // heads)
    m = (bert.BertModel if cfg.family == "bert" else nomic_bert.NomicBertModel)(cfg, "cuda", seed=1)
    ids, cu = (torch.tensor(a, dtype=torch.int32).cuda() for a in (list(range(20)), [0, 7, 8, 20]))
    every2 = lambda t: torch.stack([t, t.flip(0)], 1).flatten()[::2]
    y = m.forward(every2(ids), every2(cu), LENS)       # the loop, with heads of 64 too
    assert torch.equal(y, m.forward(every2(ids), cu, LENS)) and torch.equal(y, m.forward(ids, every2(cu), LENS))
    if heads == 2:
        assert torch.equal(y, m.forward(ids, cu, LENS))
    else:
        # other kernels: 2^-8 of a row's length at each of some twenty roundings, at random, on both sides
        assert float((y - m.forward(ids, cu, LENS)).norm(dim=1).max()) < 20 ** 0.5 * 2 ** 0.5 * 2.0 ** -8


@pytest.mark.gpu
def test_models_refuse_other_rotary_tables():
    for heads in (4, 2):
        cfg = dataclasses.replace(mc.resolve("tiny-nomic"), num_heads=heads, head_dim=D // heads)
        m = nomic_bert.NomicBertModel(cfg, "cuda", seed=1)
        ids, cu = (torch.tensor(a, dtype=torch.int32).cuda() for a in (list(range(20)), [0, 7, 8, 20]))
        t = m.cos_sin
        for bad in (t.bfloat16(), t[:, :32].contiguous(), torch.cat([t, t], 1)[:, :t.shape[1]]):
            m.cos_sin = bad
            with pytest.raises(ValueError):
                m.forward(ids, cu, LENS)


def test_embed_norm_refuses():
    _, w = _model(True)
    ids = torch.zeros(5, dtype=torch.int32)
    args = [ids, w["word"], w["type"], w["emb_ln_w"], w["emb_ln_b"], 1e-12, w["pos"], ids]
    for i, bad in ((0, ids.long()), (1, w["word"].float()), (2, w["type"][:0]), (3, w["emb_ln_w"][1:]),
                   (6, w["pos"].float()), (7, ids.long()), (7, ids[:-1]), (7, None)):
        with pytest.raises(ValueError):
            encoder.embed_norm(*args[:i], bad, *args[i + 1:])
