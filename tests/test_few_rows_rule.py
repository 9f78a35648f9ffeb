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
