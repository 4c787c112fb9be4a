"""The choice of a tile for more than 16 activation rows (csrc/gemm_t32.hip).
Host only."""
import random

import pytest
import torch  # noqa: F401  (before the library, so that the process has one HIP runtime: torch's)

import btf_hip as hip

CUS = [32, 64, 128, 256, 304]
# the tiles that are compiled: (32-row activation tiles per wave, waves along the outputs, K groups)
TILES = {(2, 4, 1), (1, 4, 1), (1, 2, 4), (1, 2, 8), (1, 1, 4), (1, 1, 8)}


def shares(K, N):
    """Shares of K in which a matrix's outputs are summed."""
    return 4 if K < 4096 or N >= 16384 else 8


@pytest.mark.parametrize("cus", CUS)
def test_every_choice_keeps_the_order_of_the_sums(cus):
    """A tile has no more K groups than any of its matrices has shares; the
    one-wave tiles and those of eight groups, which hold one share a group,
    exactly as many; a Q8 output gets whole 32-output blocks."""
    rng = random.Random(cus)
    seen = set()
    for _ in range(20000):
        mode = rng.choice(list(hip.GemvMode))
        K = 128 * rng.choice([1, 2, 4, 5, 8, 16, 31, 32, 40, 97, 136, rng.randint(1, 300)])
        N = [rng.choice([0, 1, 33, 1024, 8192, 16383, 16384, 248320, int(2 ** rng.uniform(0, 18))])
             for _ in range(2 if mode == hip.GemvMode.kSwiglu else rng.randint(1, 3))]
        if mode == hip.GemvMode.kSwiglu:
            N[1] = N[0]
        M = int(2 ** rng.uniform(4.1, 12))
        q8 = M <= 32 and (mode == hip.GemvMode.kSwiglu or len(N) == 1) and N[0] % 32 == 0 and rng.random() < 0.5
        tile = hip.gemm_tile(cus, N, K, M, mode, q8)
        if not any(N):
            assert tile is None
            continue
        assert tile in TILES
        seen.add(tile)
        mt, wn, wk = tile
        used = {shares(K, n) for n in (N[:1] if mode == hip.GemvMode.kSwiglu else N) if n}
        if (wn, wk) in ((1, 4), (1, 8), (2, 8)):
            assert used == {wk}, (N, K, M, mode)
        else:
            assert wk <= min(used)
        if q8:
            assert mt == 1 and wn * (16 if mode == hip.GemvMode.kSwiglu else 32) % 32 == 0
    assert seen == TILES


@pytest.mark.parametrize("cus", CUS)
@pytest.mark.parametrize("K", [256, 1024, 3968, 4096, 5120])
def test_tile_follows_tiles_per_cu(cus, K):
    """The lines lie at counts of 32 x 32 tiles per CU."""
    def at(tiles, M=32):  # so many tiles of one row group, over as many segments as keep N below 16384
        n = [tiles // 3 * 32, tiles // 3 * 32, (tiles - 2 * (tiles // 3)) * 32]
        return hip.gemm_tile(cus, n, K, M)
    few, one, two, four = (1, 1, 8 if K >= 4096 else 4), (1, 4, 1), (1, 2, 8), (1, 2, 4)
    assert at(cus) == few and at(10 * cus + 1) == one
    assert at(cus + 1) == (few if K <= 512 else two if K >= 4096 else four)
    if K <= 512:
        assert at(4 * cus - 1) == few and at(4 * cus) == one
    elif cus < 256:  # (more tiles than 16384 outputs a segment have four shares)
        assert at(2 * cus) == (two if K >= 4096 else four) and at(2 * cus + 1) == four and at(10 * cus) == four
    assert at(16 * cus, 64) == (2, 4, 1) and at(16 * cus - 1, 64) == one


def test_no_tile_for_few_rows():
    assert hip.gemm_tile(256, [5120], 5120, 16) is None
    assert hip.gemm_tile(256, [5120], 100, 32) is None
