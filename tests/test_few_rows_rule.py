"""The rule that sends one or two rows to K25 (ops.gemv_splits): what it takes and what it leaves."""
import pytest
import torch

from llm_mcp_amd import ops


def _rows(M, K, ld=None, offset=0):
    """M rows of K at a stride of ld, the first one ``offset`` elements past a 16-byte boundary."""
    n = M * (ld or K)
    buf = torch.zeros(n + offset + 8, dtype=torch.bfloat16)
    at = -buf.data_ptr() // 2 % 8 + offset
    return buf[at:at + n].view(M, ld or K)[:, :K]


@pytest.mark.parametrize("M,N,K,epi,splits", [
    (1, 32, 1024, 0, 1), (2, 6144, 4096, 0, 1), (1, 128256, 2048, 0, 1), (1, 16384, 2048, 3, 1),
    (2, 2048, 8192, 2, 2), (1, 2048, 3072, 2, 1), (1, 4096, 8192, 2, 1), (1, 64, 1024, 4, 1),
    (0, 64, 1024, 0, None), (3, 64, 1024, 0, None), (1, 48, 1024, 0, None), (1, 64, 1536, 0, None)])
def test_shapes(M, N, K, epi, splits):
    assert ops.gemv_splits(torch.zeros(M, K).bfloat16(), torch.empty(N, K, dtype=torch.bfloat16), epi) == splits


def test_layouts():
    w, x = _rows(64, 1024), _rows(2, 1024)
    assert ops.gemv_splits(x, w) == 1
    assert ops.gemv_splits(_rows(2, 1024, 1032), _rows(64, 1024, 2048)) == 1      # strided rows
    assert ops.gemv_splits(x.float(), w) is None and ops.gemv_splits(x, w.float()) is None
    assert ops.gemv_splits(_rows(2, 1024, 1028), w) is None                       # rows off 16 bytes
    assert ops.gemv_splits(_rows(2, 1024, offset=4), w) is None
    assert ops.gemv_splits(x, _rows(1024, 64).t()) is None                        # columns apart
    assert ops.gemv_splits(x.flip(0).t().contiguous().t(), w) is None
    assert ops.gemv_splits(x, w, 0, _rows(2, 64, 66)) == 1                        # any even row of output
    assert ops.gemv_splits(x, w, 0, _rows(2, 64, 67)) is None
    assert ops.gemv_splits(x, w, 0, _rows(2, 64, 66, offset=1)) is None
    assert ops.gemv_splits(x, w, 0, _rows(64, 2).t()) is None


@pytest.mark.parametrize("step", [2, 4])
def test_operands_and_destinations(step):
    """What K25 and K23 leave to the routes that stood before them: other types, layouts and devices,
    destinations that they cannot write whole or that are read meanwhile, empty products."""
    x, w = _rows(2, 1024), _rows(64, 1024)
    ok = lambda *a, **k: ops.few_rows_ok(*a, **k, step=step)
    assert ok(x, w) and ok(x, w, 0, _rows(1, 64)[0], _rows(2, 64, 72))
    assert ok(x, w, 3, None, _rows(2, 32, 36)) and not ok(x, w, 3, None, _rows(2, 64))
    assert not ok(x, w, 0, torch.zeros(64)) and not ok(x, w, 0, _rows(1, 32)[0])
    assert not ok(_rows(2, 512), w)
    assert not ok(x, w[:0]) and not ok(x[:, :0], w[:, :0])
    for out in (torch.zeros(2, 64), _rows(2, 64, 65), _rows(2, 64, offset=1), _rows(64, 2).t(),
                _rows(1, 64).expand(2, 64), _rows(3, 64), torch.empty(2, 64, dtype=torch.bfloat16, device="meta")):
        assert not ok(x, w, 0, None, out)
    assert ok(x, w, 0, None, _rows(2, 64, 66)) == (step == 2)
    assert ok(x, w, 0, None, _rows(2, 64, offset=2)) == (step == 2)
    assert not ok(x, w, 0, None, x[:, :64]) and not ok(x, w, 0, None, w[:2, :64])      # read meanwhile
    assert not ok(x, w.to("meta"))


def test_gradients_and_transforms():
    x, w = _rows(2, 1024), _rows(64, 1024)
    g = w.clone().requires_grad_()
    assert not ops.few_rows_ok(x, g) and not ops.few_rows_ok(x.clone().requires_grad_(), w)
    with torch.no_grad():
        assert ops.few_rows_ok(x, torch.nn.Parameter(w))
    assert ops.few_rows_ok(x, torch.nn.Parameter(w, requires_grad=False))
    seen = []
    torch.vmap(lambda a: (seen.append(ops.few_rows_ok(a, w)), a)[1])(x[None])
    with torch._subclasses.fake_tensor.FakeTensorMode() as mode:
        seen.append(ops.few_rows_ok(torch.empty(2, 1024, dtype=torch.bfloat16), mode.from_tensor(w)))
    with torch.autograd.forward_ad.dual_level():
        seen.append(ops.few_rows_ok(torch.autograd.forward_ad.make_dual(x, x), w))
    assert seen == [False] * 3


@pytest.mark.parametrize("M,N,K,epi,splits", [
    (32, 2048, 2048, 0, 1), (33, 2048, 2048, 0, None), (32, 32, 1152, 0, 1), (24, 64, 1280, 0, 1),
    (25, 64, 1280, 0, None), (32, 64, 1280, 3, 1), (17, 64, 2080, 0, None), (16, 64, 4096, 0, 1),
    (9, 64, 4128, 0, None), (8, 64, 5120, 0, 1), (1, 64, 5152, 0, None), (8, 512, 4096, 3, 1),
    (9, 512, 4096, 4, None), (32, 4096, 256, 0, 1), (1, 4128, 480, 0, None), (32, 6144, 768, 0, 1),
    (1, 6144, 1056, 0, None), (32, 12288, 256, 3, 1), (1, 12320, 256, 3, None), (3, 3072, 4096, 0, None),
    (32, 64, 14336, 2, 4), (32, 1024, 6144, 2, 4), (32, 2048, 2048, 2, 2), (17, 2304, 2560, 2, None),
    (16, 2304, 2560, 2, 1), (8, 4096, 4096, 2, 1), (9, 4096, 4096, 2, None), (8, 2560, 4608, 2, None),
    (8, 6144, 2048, 2, 1), (8, 6144, 2560, 2, None), (8, 12288, 1280, 2, None), (9, 6144, 1056, 2, None),
    (3, 96, 48, 0, None), (3, 48, 96, 0, None), (0, 96, 96, 0, None)])
def test_shapes_of_k23(M, N, K, epi, splits):
    assert ops.sgemm_splits(M, N, K, epi) == splits


def test_products_that_the_table_keeps(monkeypatch):
    """Shapes whose table kernel was measured faster: they have one, and neither kernel takes them."""
    keep, taken = ops._keep_table(), 0
    cases = [(M, *k) for k, ranges in keep.items() for a, b in ranges for M in range(a, b + 1)]
    assert cases and all(1 <= M <= ops.SGEMM_MAX_M and ops.dgemm_choice(M, *k) for M, *k in cases)
    for off in (False, True):
        if off:
            monkeypatch.setattr(ops, "_KEEP_TABLE", {})
        for M, N, K, epi in cases:
            x, w = torch.zeros(M, K).bfloat16(), torch.empty(N, K, dtype=torch.bfloat16, device="meta")
            got = ops.gemv_splits(x, w, epi), ops.sgemm_splits(M, N, K, epi)
            assert off or got == (None, None)
            taken += got != (None, None)
    assert taken == len(cases)               # without the list one of them takes each
