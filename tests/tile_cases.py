"""Sizes that reach every tile of mfma_tiles.hpp's list, looked up in the built library: a list by hand goes stale with the costs that the tile is picked by."""
import functools
import os
import re

ROWS = (1, 5, 17, 33, 40, 66, 70, 97, 130, 195, 257, 263, 321, 391, 481, 641, 769, 866, 963, 1063, 1375, 1859, 2029, 2507, 3001, 4003)
COLUMNS = (32, 96, 160, 288, 544, 992, 1568, 2336, 3232, 4128, 4896, 5408, 5920, 6560, 7200, 7840, 9056, 10400)


@functools.lru_cache(maxsize=None)
def tiles():
    """(rows / 16, columns / 64, chunks in flight) in their order."""
    from vllmini_amd import build

    text = open(os.path.join(build.CSRC, "mfma_tiles.hpp")).read()
    body = text[text.index("constexpr Tile TILES[]"):]
    return tuple(tuple(map(int, t)) for t in re.findall(r"\{(\d+), (\d+), (\d+),", body[: body.index(";")]))


def places():
    """Every tile with every number of chunks of K that its walk may leave behind its whole rounds."""
    return [(i, left) for i, (_, _, d) in enumerate(tiles()) for left in range(1, d + 1)]


@functools.lru_cache(maxsize=None)
def size_for(tile, left, groups=(1,), most_chunks=40):
    """(M, N, K, groups), N a multiple of 32: the cheapest product that the list's rule gives to the tile, with rows and columns left over and so many chunks of K left behind two
    rounds of its walk or more; None where none of these sizes does."""
    from vllmini_amd import hybrid_ops

    pick, (mi, ni, d), best = hybrid_ops.load().vmi_hy_tiles_pick, tiles()[tile], None
    for g in groups:
        for chunks in range(2 * d + left, most_chunks, d):
            for M in ROWS:
                for N in COLUMNS:
                    cost = M * N * chunks * g
                    if M % (16 * mi) and N % (64 * ni) and (best is None or cost < best[0]) and pick(M, N, 64 * chunks, g) == tile:
                        best = cost, (M, N, 64 * chunks, g)
    return best and best[1]
