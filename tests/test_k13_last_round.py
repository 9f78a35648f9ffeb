"""K13's last, partly filled round of tiles in pieces along K (csrc/kernels/pgemm.hip): the cut as the
kernel walks it, on the host."""
import collections

import pytest

from llm_mcp_amd import native

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
                    assert not mine & slabs and min(mine) >= 0 and max(mine) < row * 16
                    slabs |= mine


def test_uncut_products_have_no_pieces():
    """Fewer than 8 workgroups among them."""
    for ntiles in (1, 3, 7, 8, 255, 256, 300):
        assert _pieces(ntiles, 12, 0, min(ntiles, CUS)) == []
