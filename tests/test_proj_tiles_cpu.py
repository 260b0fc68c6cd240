"""The sizes of the GPU tests that are meant to reach each tile of the
projection still do (a change of the cost table moves them)."""

import pytest

from tests.proj_tiles import BATCH_SIZES, COSTS, PACKED_SIZES, TILES, choose_tile, in_proj_columns, ragged


def test_tables_are_read():
    assert [c[0] for c in COSTS] == list(TILES) and len(TILES) == 12
    assert TILES["Tile256x256"] == (256, 253, 2) and TILES["Tile32x32"] == (32, 29, 3)


@pytest.mark.parametrize("tile,rows,H,dv,D,ck", PACKED_SIZES)
def test_packed_sizes(tile, rows, H, dv, D, ck):
    lengths = ragged(rows)
    assert sum(lengths) + 3 * len(lengths) == rows and min(lengths) >= 0 and len(lengths) <= 256
    assert choose_tile(rows, D, in_proj_columns(H, 128, dv)) == tile


@pytest.mark.parametrize("tile,B,T,H,dv,D,ck", BATCH_SIZES)
def test_batch_sizes(tile, B, T, H, dv, D, ck):
    assert choose_tile(B * (T + 3), D, in_proj_columns(H, 128, dv)) == tile


def test_every_tile_is_reached():
    for sizes in (PACKED_SIZES, BATCH_SIZES):
        assert {s[0] for s in sizes} == set(TILES)
