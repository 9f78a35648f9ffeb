"""The encoders' choice of a product's kernel (csrc/kernels/encoder.hip enc_plan), on the host."""
import dataclasses

import pytest
import torch

from llm_mcp_amd import native, ops
from llm_mcp_amd.models import config as mc
from llm_mcp_amd.ops import encoder

SMALL, K13 = 100, -1            # EncPlan's cfg for K23 and K13


@pytest.mark.parametrize("cus", [32, 64, 128, 256])
@pytest.mark.parametrize("d,I", [(256, 256), (768, 3072), (1024, 4096), (1792, 4864), (2048, 14336)])
@pytest.mark.parametrize("gelu", [True, False])
def test_plans_are_what_the_kernels_take(cus, d, I, gelu):
    """Every product of a layer from one row to 64 k: tiles divide the columns, K slices are whole
    steps and as many as the norm sums, pair epilogues have whole pairs a wave, and the tiles that
    add a bias are those of dgemm.hip's dg_bias_tile."""
    rows = [1, 2, 16, 31, 32, 33, 64, 65, 127, 128, 129, 255, 256, 257, 300, 500, 777, 1000, 1500, 2048, 3000,
            5000, 8192, 11760, 19153, 32768, 65536]
    for M in rows:
        for N, K, act, partials in ((3 * d, d, 0, False), (d, d, 0, True),
                                    (I if gelu else 2 * I, d, 4 if gelu else 3, False), (d, I, 0, True)):
            cfg, s = native.kernels().enc_plan(M, N, K, act, partials, cus)
            if cfg == K13:
                assert N % 256 == 0 and K % 64 == 0 and K >= 192
            elif cfg == SMALL:
                assert not partials and s == 1 and M <= 32 and N % 32 == 0 and K % 32 == 0
            else:
                bm, bn = ops.DGEMM_CONFIGS[cfg]
                bk = 128 if cfg in ops.DGEMM_BK128 else 64
                assert N % bn == 0 and K % (bk * s) == 0 and s in (1, 2, 3, 4, 6, 8, 12, 16)
                assert partials or s == 1
                assert act != 3 or ops.swiglu16_ok(cfg)
                assert (bm <= 128 and bn <= 128) if bk == 128 else (bm, bn) == (128, 256)


@pytest.mark.parametrize("cus", [32, 256])
def test_rounds_are_of_the_device(cus):
    """One round of 64 x 64 tiles on the device at hand is not cut into slices that make it two."""
    for M in (64, 128, 192, 256):
        cfg, s = native.kernels().enc_plan(M, 1024, 4096, 0, True, cus)
        if cfg >= 0 and cfg != SMALL:
            bm, bn = ops.DGEMM_CONFIGS[cfg]
            assert -(-M // bm) * (1024 // bn) * s <= max(cus, -(-M // bm) * (1024 // bn))


# rows of a request between which every kernel, tile and slice that the choice has for a product
# of the model up to 8,192 rows occurs
ROWS = {"nomic-embed-text": [1, 65, 155, 193, 321, 449, 641, 897, 1345, 1793, 2689, 3585, 4030, 5377, 5441],
        "mxbai-embed-large": [1, 75, 129, 156, 321, 513, 641, 668, 1345, 2689, 4097]}


def _plans(cfg, M):
    d, I, gelu = cfg.hidden_size, cfg.intermediate_size, cfg.family == "bert"
    return {(i, *native.kernels().enc_plan(M, *x, 256)) for i, x in enumerate(
        ((3 * d, d, 0, False), (d, d, 0, True), (I if gelu else 2 * I, d, 4 if gelu else 3, False),
         (d, I, 0, True)))}


@pytest.mark.parametrize("model", ROWS)
def test_rows_below_reach_every_plan(model):
    cfg = mc.resolve(model)
    every = set().union(*(_plans(cfg, M) for M in range(1, 8193)))
    assert set().union(*(_plans(cfg, M) for M in ROWS[model])) == every


@pytest.mark.gpu
@pytest.mark.parametrize("model,rows", [(m, r) for m in ROWS for r in ROWS[m]])
def test_every_plan_against_the_models_own_loop(model, rows):
    """One layer of the model's sizes on every kernel, tile and slice that it is planned on: the
    vectors of the loop over single ops, which runs K13 alone."""
    from llm_mcp_amd.models.bert import BertModel
    from llm_mcp_amd.models.nomic_bert import NomicBertModel
    cfg = dataclasses.replace(mc.resolve(model), num_layers=1)
    m = (BertModel if cfg.family == "bert" else NomicBertModel)(cfg, "cuda", seed=4)
    g = torch.Generator().manual_seed(rows)
    longest, lens = 500, []
    while sum(lens) < rows:
        lens.append(min(rows - sum(lens), longest))
    ids = torch.randint(0, 30000, (rows,), generator=g, dtype=torch.int32).cuda()
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32).cuda()
    calls = encoder.LAYER_CALLS[0]
    a = m.forward(ids, cu, lens)
    assert encoder.LAYER_CALLS[0] == calls + 1
    keep, encoder.layers_ok = encoder.layers_ok, lambda *x: None
    try:
        b = m.forward(ids, cu, lens)
    finally:
        encoder.layers_ok = keep
    # bf16 rows through one layer and its two norms: 2^-8 of a row's length at each of some ten
    # roundings, at random, against the other's
    assert float((a - b).norm(dim=1).max()) < 10 ** 0.5 * 2 ** 0.5 * 2.0 ** -8
