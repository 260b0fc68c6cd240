"""Which tile the projection's launch picks (choose_tile in proj.hip), restated
over the tables in the sources, so that the sizes of tests that are meant to
reach a tile can be checked on the CPU; and those sizes."""

import os
import re

import numpy as np

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gdn_18646_amd", "csrc")


def _read(name):
    with open(os.path.join(CSRC, name)) as f:
        return f.read()


# tile -> its template arguments (CW, TW, WMT, WNT, NS, PER_CU, PHASED, KS, KD)
ARGS = {}
for _name, _args in re.findall(r"using (Tile\w+) = ProjTile<([^>]*)>", _read("proj_mfma.hpp")):
    _args = [{"true": 1, "false": 0}.get(x.strip(), x) for x in _args.split(",")]
    ARGS[_name] = tuple(int(x) for x in _args) + (0, 1, 1)[len(_args) - 6:]
# tile -> (columns, tokens written, K stages in LDS), and the costs in the launch's order
TILES = {name: (16 * cw * wmt, 16 * tw * wnt - 3, ns) for name, (cw, tw, wmt, wnt, ns, *_) in ARGS.items()}
COSTS = [(name, *(np.float32(x) for x in cost)) for name, *cost in re.findall(
    r"cost_of<(Tile\w+)>\(([\d.]+)f, ([\d.]+)f, ([\d.]+)f, ([\d.]+)f\)", _read("proj.hip"))]


def choose_tile(rows, D, D_out):
    """rows: 3 cache rows and the tokens of every sequence."""
    nk, best = np.float32(D // 64), None
    for name, a1, b1, a2, b2 in COSTS:
        cols, outs, _ = TILES[name]
        n = -(-(-(-rows // outs) * -(-D_out // cols)) // 256)
        us = np.float32(n // 2) * (a2 + b2 * nk) + np.float32(n % 2) * (a1 + b1 * nk)
        if best is None or us < best[0]:
            best = (us, name)
    return best[1]


def in_proj_columns(H, dk, dv):
    return 2 * H * dk + H * dv + 2 * H


def ragged(rows):
    """Sequence lengths that make exactly `rows` rows with their 3 cache rows
    each: empty ones, ones shorter than the conv window, and ones that end
    around a wave's, a tile's or a chunk's worth of rows."""
    lengths, cycle, i = [], (0, 1, 2, 3, 29, 5, 61, 0, 17, 125, 4, 253), 0
    while rows > 0:
        n = cycle[i % len(cycle)]
        if rows - n - 3 < 3:
            n = rows - 3
        lengths.append(n)
        rows -= n + 3
        i += 1
    return lengths


# (tile, rows, H, dv, D, conv taps) of the packed in-projection, dk = 128; the K
# of the first eight is no longer than the tile's ring holds or one stage more.
# (128 x 160, 128 x 128 with four stages and 64 x 128 are not chosen for a K as
# short as their rings.)
PACKED_SIZES = [
    ("Tile256x256", 2520, 16, 128, 64, 4), ("Tile256x224", 2880, 16, 256, 64, 3), ("Tile256x192", 880, 32, 128, 64, 4),
    ("Tile256x160", 880, 16, 256, 192, 2), ("Tile128x128", 92, 16, 256, 64, 4), ("Tile64x64Wide", 32, 16, 256, 64, 4),
    ("Tile64x64", 92, 16, 256, 128, 4), ("Tile64x32", 62, 16, 256, 64, 3), ("Tile32x32", 40, 4, 128, 64, 4),
    ("Tile32x32", 40, 4, 128, 192, 2), ("Tile64x32", 62, 16, 256, 320, 4), ("Tile128x160", 380, 16, 256, 320, 4),
    ("Tile128x128Deep", 188, 16, 256, 2048, 4), ("Tile64x128Deep", 1240, 4, 128, 448, 3),
    ("Tile256x160", 880, 16, 256, 448, 4), ("Tile256x256", 1600, 16, 256, 512, 2)]

# (tile, B, T, H, dv, D, conv taps) of batches of equal lengths with caches.
BATCH_SIZES = [
    ("Tile256x256", 4, 627, 16, 128, 64, 4), ("Tile256x224", 3, 957, 16, 256, 64, 4), ("Tile256x192", 4, 217, 32, 128, 64, 4),
    ("Tile256x160", 2, 437, 16, 256, 192, 4), ("Tile128x128", 4, 20, 16, 256, 64, 2), ("Tile64x64Wide", 4, 5, 16, 256, 64, 4),
    ("Tile64x64", 23, 1, 16, 256, 128, 4), ("Tile64x32", 2, 28, 16, 256, 64, 4), ("Tile32x32", 5, 5, 4, 128, 64, 3),
    ("Tile128x160", 4, 92, 16, 256, 320, 4), ("Tile128x128Deep", 2, 91, 16, 256, 2048, 4),
    ("Tile64x128Deep", 5, 245, 4, 128, 448, 4)]
