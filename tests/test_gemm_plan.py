"""The tile rules of the FP8, NVFP4 and BF16 GEMMs, evaluated on the host."""
from __future__ import annotations

import ctypes as C

import pytest

from qw38_amd._lib import QW38_INVALID_ARGUMENT, lib

CUS = 256
FP8, NVFP4, NVFP4_PAIRED, BF16, BF16_PAIRED, BF16_UNALIGNED, BF16_PAIRED_UNALIGNED = range(7)


def plan(path, n, m):
    p = (C.c_uint32 * 3)()
    assert lib().qw38_gemm_plan(path, n, m, CUS, p) == 0
    return p[0], p[1], p[2]


@pytest.mark.parametrize("path,step,top", [(FP8, 128, 12288), (NVFP4, 136, 17408), (NVFP4_PAIRED, 136, 17408),
                                           (BF16, 248, 36000), (BF16_PAIRED, 248, 18000),
                                           (BF16_UNALIGNED, 248, 36000), (BF16_PAIRED_UNALIGNED, 248, 18000)])
def test_every_tile_is_chosen(path, step, top):
    """No rule carries a tile that nothing in the entry's range takes."""
    last = 1024 if path < BF16 else 4096
    tokens = list(range(1, 257, 15)) + list(range(257, last + 1, 41)) + [last]
    seen = set()
    for n in range(step, top + 1, step):
        for m in tokens:
            _, tile, tiles = plan(path, n, m)
            seen.add(tile)
    assert seen == set(range(tiles))


@pytest.mark.parametrize("n,m,tile", [(12288, 40, 3), (12288, 64, 3), (9216, 64, 3), (6912, 80, 3), (9216, 24, 5),
                                      (12288, 16, 4), (12288, 512, 1), (12288, 1024, 0)])
def test_fp8_choice_is_the_fastest(n, m, tile):
    """Where the 64 x 16 tile takes 20 to 27% more than the measured best (its
    blocks beyond the first on a CU cost more than its rule said), and where it
    or the largest tiles are the best."""
    assert plan(FP8, n, m)[1] == tile


def test_gpu_sizes_take_every_tile():
    """The GPU tests that compare tiles run all of them."""
    import test_gpu_fp8
    import test_gpu_nvfp4
    for path, sizes in ((FP8, test_gpu_fp8.GEMM_SIZES), (NVFP4, test_gpu_nvfp4.GEMM_SIZES),
                        (NVFP4_PAIRED, test_gpu_nvfp4.GEMM_SIZES)):
        seen = {plan(path, n, m)[1] for n, ms in sizes for m in ms}
        assert seen == set(range(plan(path, 128, 1)[2])), path


def test_refusals():
    p = (C.c_uint32 * 3)()
    for args in ((7, 128, 1, CUS, p), (0, 0, 1, CUS, p), (0, 128, 0, CUS, p), (0, 128, 1, 0, p), (0, 128, 1, CUS, None)):
        assert lib().qw38_gemm_plan(*args) == QW38_INVALID_ARGUMENT


@pytest.mark.parametrize("path,n,m", [(BF16, 17408, 768), (BF16, 5120, 3072), (BF16, 12288, 4096), (BF16, 8704, 1792),
                                      (BF16_PAIRED, 17408, 4096), (BF16_PAIRED, 17408, 3072), (BF16_PAIRED, 5120, 1536)])
def test_big_tiles_where_ring_tiles_lose(path, n, m):
    """A grid of 256-row tiles whose last round is nearly full, and paired grids
    of many rounds, run on them (on ring tiles alone they take 10 to 30% more)."""
    assert plan(path, n, m)[0] > 0


@pytest.mark.parametrize("n,m", [(248320, 150), (248320, 129), (248320, 2048)])
def test_one_launch_where_two_gain_nothing(n, m):
    """Big tiles on whole rounds with ring tiles behind are taken where they gain
    more than 1%: the second launch's start and end cost as much (2 to 18% of a short K)."""
    assert plan(BF16, n, m)[0] * 256 >= n
