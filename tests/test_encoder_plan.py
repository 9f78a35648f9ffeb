"""The encoders' choice of a product's kernel (csrc/kernels/encoder.hip enc_plan), on the host."""
import pytest

from llm_mcp_amd import native, ops

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
