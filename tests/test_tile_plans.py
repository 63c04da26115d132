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
