"""bf16 prefill in tiles of 32, 64 and 128 rows (k_gemm_tile_short; run on an MI355X): every tile
height's edges, K split and not, X staged, read in place and rounded on the way."""

import numpy as np
import pytest

from oracle import mtc_oracle as O
from tensorpack_amd.kernels.gemm import mtc_gemm_group

from conftest import cell_format_matrices, leaf_matrix, tile_rows

pytestmark = pytest.mark.gpu

# (K, N): a partial last K-step and column tile; one K-step; many K-steps (split K, several per block)
SHAPES = {"ragged": (992, 288), "one": (64, 256), "deep": (4096, 544)}


@pytest.fixture(scope="module")
def mats():
    return cell_format_matrices(SHAPES)


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("form", ["qt", "qtp", "p16", "uniform"])
@pytest.mark.parametrize("x", ["fp32", "bf16"])
def test_short_tiles_at_every_height(gpu, mats, shape, form, x):
    import torch
    m, W_hat = mats[shape, form]
    K = W_hat.shape[0]
    t = m.device_tiles(gpu)
    Wb = torch.from_numpy(np.ascontiguousarray(W_hat, np.float32)).bfloat16().double().numpy()
    for M in (1, 17, 31, 32, 33, 64, 65, 100, 128, 129, 250, 256):
        print("short prefill", shape, form, x, M, flush=True)
        X = torch.from_numpy(np.random.RandomState(M).randn(M, K).astype(np.float32))
        ref = X.bfloat16().double().numpy() @ Wb
        Xg = (X if x == "fp32" else X.bfloat16()).to(gpu)
        Y = t.gemm_bf16(Xg, out_dtype=torch.float32)
        # products of bf16 values are exact in fp32: K roundings to fp32 on the way at most (a random walk of half ulps)
        err = O.relative_frobenius_error(ref, Y.cpu().numpy())
        assert err <= np.sqrt(K) * 2.0 ** -24, (M, err)
        assert torch.equal(t.gemm_bf16(Xg, out_dtype=torch.bfloat16), Y.bfloat16())   # the same sums, rounded once
        # a group's members split K as the single call does: the same sums in the same order
        for Z in mtc_gemm_group(Xg, [m, m], compute="bf16"):
            assert torch.equal(Z, Y), M


@pytest.mark.parametrize("form", ["qt", "qtp", "uniform"])
@pytest.mark.parametrize("x", ["fp32", "bf16"])
def test_128_row_tiles(gpu, form, x):
    """Sizes that take 128-row tiles, the last of 72 rows, with K split: a single call (X in place, staged or rounded
    on the way), a group and a batch (which run the height of the single calls)."""
    import torch
    from tensorpack_amd.device import GemmBatch
    K, N, M = 1504, 5472, 200
    m, W_hat = leaf_matrix(form, K, N, 7)
    t = m.device_tiles(gpu)
    assert tile_rows(t, M, False) == 128
    print("128-row tiles", form, x, flush=True)
    X = torch.from_numpy(np.random.RandomState(M).randn(M, K).astype(np.float32)).to(gpu)
    ref = X.bfloat16().double() @ torch.from_numpy(W_hat).to(gpu).bfloat16().double()
    Xg = X if x == "fp32" else X.bfloat16()
    Y = t.gemm_bf16(Xg, out_dtype=torch.float32)
    assert ((Y - ref).norm() / ref.norm()).item() <= np.sqrt(K) * 2.0 ** -24      # as above
    assert torch.equal(t.gemm_bf16(Xg, out_dtype=torch.bfloat16), Y.bfloat16())
    for Z in mtc_gemm_group(Xg, [m, m], compute="bf16"):
        assert torch.equal(Z, Y)
    for Z in GemmBatch([t, t.clone()], [Xg, Xg]).launch():
        assert torch.equal(Z, Y)
