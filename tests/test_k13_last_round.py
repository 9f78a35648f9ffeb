"""K13's last, partly filled round of tiles in pieces along K (csrc/kernels/pgemm.hip): the cut as the
kernel walks it, on the host."""
import collections

import pytest
import torch

from llm_mcp_amd import native, ops

CUS = 256


def _pieces(ntiles, nk, share, cus=CUS):
    return [dict(zip(("wg", "tile", "kb", "ke", "slab", "p", "of"), x))
            for x in native.kernels().pgemm_last_round(cus, ntiles, nk, share)]


@pytest.mark.parametrize("cus", [32, 64, 256])
@pytest.mark.parametrize("nk", [8, 12, 13, 64, 224])
def test_pieces_cover_the_round(cus, nk):
    """Every K-step of every tile of the round in one piece, a workgroup at most in a piece of a tile,
    the pieces of a tile in K order on slabs of their own, whatever the number of tiles."""
    row = cus // 8
    for rest in {1, 2, row - 1, row, row + 1, 3 * row, 4 * row + 1, 7 * row - 1, 7 * row}:
        most = -(-rest // row)
        for share in range(most + 1, 9):
            if most * nk // share < 4:
                continue
            ps = _pieces(2 * cus + rest, nk, share, cus)
            tiles, slabs = collections.defaultdict(list), set()
            for q in ps:
                tiles[q["tile"]].append(q)
                assert 0 <= q["kb"] < q["ke"] <= nk and 0 <= q["wg"] < cus
            assert sorted(tiles) == list(range(2 * cus, 2 * cus + rest))
            for t in tiles.values():
                t.sort(key=lambda q: q["kb"])
                assert [q["p"] for q in t] == list(range(len(t))) and {q["of"] for q in t} == {len(t)}
                assert t[0]["kb"] == 0 and t[-1]["ke"] == nk
                assert all(a["ke"] == b["kb"] for a, b in zip(t, t[1:]))
                assert len({q["wg"] for q in t}) == len(t)
                if len(t) > 1:
                    assert [q["slab"] - t[0]["slab"] for q in t] == list(range(len(t)))
                    mine = {q["slab"] for q in t}
                    assert not mine & slabs and min(mine) >= 0 and max(mine) < min(rest, row) * (share + most - 1)
                    slabs |= mine


def test_uncut_products_have_no_pieces():
    """Fewer than 8 workgroups among them."""
    for ntiles in (1, 3, 7, 8, 255, 256, 300):
        assert _pieces(ntiles, 12, 0, min(ntiles, CUS)) == []


@pytest.mark.parametrize("cus", [32, 256])
def test_scratch_holds_the_pieces_and_little_more(cus):
    """The slabs of a product: a row's parts and one more for each of its tiles after the first, for as
    many rows as there are tiles for; every piece that is joined inside them."""
    plan, cut = native.kernels().pgemm_tail_plan, 0
    for M in (1, 100, 257, 600, 2048, 2300, 6464, 7680):
        for N in (256, 512, 768, 4096, 6144, 18688, 28672):
            for K in (192, 768, 2048, 4096, 8192, 14336):
                share, floats = plan(M, N, K, cus)
                assert (share == 0) == (floats == 0)
                if not share:
                    continue
                cut += 1
                tiles = -(-M // 256) * (N // 256)
                ps = _pieces(tiles, K // 64, share, cus)
                joined = [q["slab"] for q in ps if q["of"] > 1]
                assert not joined or max(joined) * 65536 < floats
                rest, row = tiles % cus, cus // 8
                assert floats == 65536 * min(rest, row) * (share - 1 + -(-rest // row))
    assert cut > 20
    assert plan(100, 256, 8192, 256) == (4, 4 * 65536)                 # one tile: 1 MB
    assert plan(2048, 4096, 4096, 0) == plan(2048, 4096, 4096, 250) == (0, 0)


def test_whole_tiles_where_no_memory_is_left(monkeypatch):
    def full(*a, **k):
        raise torch.cuda.OutOfMemoryError("out of memory")
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(ops, "pgemm_counters", lambda dev: "counters")
    slabs, counters = ops.pgemm_tail_memory(torch.device("cpu"), 12)
    assert slabs.numel() == 12 and counters == "counters"
    assert ops.pgemm_tail_memory(torch.device("cpu"), 0) == (None, None)
    monkeypatch.setattr(torch, "empty", full)
    assert ops.pgemm_tail_memory(torch.device("cpu"), 12) == (None, None)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    assert ops.pgemm_tail_memory(torch.device("cpu"), 12) == (None, None)
