"""The tile kernels' choice of rows per tile and K splits (mtc_tile_plan, host only)."""

import ctypes
import math
import random

import pytest

from tensorpack_amd import _abi, _native

CUS, XCDS = 256, 8


@pytest.fixture(scope="module")
def plan():
    lib = _native.hip_lib()

    def of(M, K, N, fp32):
        d = _abi.MtcTileDesc()
        d.abi_version, d.K, d.N, d.n_ksteps, d.n_col_tiles = _abi.ABI_VERSION, K, N, -(-K // 64), -(-N // 256)
        d.payload_dwords, d.cells, d.step_off, d.payload = 64, 0x1000, 0x1000, 0x1000
        rows, splits = ctypes.c_int32(), ctypes.c_int32()
        assert lib.mtc_tile_plan(ctypes.byref(d), M, int(fp32), ctypes.byref(rows), ctypes.byref(splits)) == 0
        return rows.value, splits.value
    return of


def _shapes(n, lo, hi, seed):
    rng = random.Random(seed)
    size = lambda a, b: round(math.exp(rng.uniform(math.log(a), math.log(b))))
    for _ in range(n):
        yield size(lo, hi), 32 * size(8, 192), 32 * size(8, 192)


def _one_round_of_the_chip_only(M, N, rows, splits):
    """Blocks that fit one round of the chip's CUs, but not one of the XCD that gets the most tiles (an XCD runs
    every eighth tile, all its splits)."""
    tiles = -(-M // rows) * -(-N // 256)
    return tiles * splits <= CUS and -(-tiles // XCDS) * splits > CUS // XCDS


def test_f32_plan_counts_rounds_on_the_fullest_xcd(plan):
    for M, K, N in [(545, 1664, 4224), (155, 2464, 2816)] + list(_shapes(3000, 17, 1024, 1)):
        assert not _one_round_of_the_chip_only(M, N, *plan(M, K, N, True)), (M, K, N, plan(M, K, N, True))


def test_tall_bf16_plans_keep_their_pricing(plan):
    """Calls of more than 256 rows: 2 us a K-step, partials at 4 bytes a picosecond and 3 us for their reduction.
    Shapes that a dearer block splits sooner and slower stay unsplit."""
    for M, K, N in ((339, 352, 3040), (466, 416, 1888), (409, 416, 2400), (443, 512, 3168), (465, 768, 6048)):
        assert plan(M, K, N, False) == (256, 1), (M, K, N)
    for M, K, N in _shapes(2000, 257, 4096, 2):
        tiles, steps = -(-M // 256) * -(-N // 256), -(-K // 64)
        best = (1e300, 1)
        for s in range(1, 1 if tiles >= CUS else 1 + max(1, min(-(-CUS // tiles), steps // 2))):
            per = -(-steps // s)
            s = -(-steps // per)
            rounds = -(-(-(-tiles // XCDS) * s) // (CUS // XCDS))
            best = min(best, (rounds * per * 2.0 + (s * 8.0 * M * N / 4e6 + 3.0 if s > 1 else 0.0), s))
        assert plan(M, K, N, False) == (256, best[1]), (M, K, N)
