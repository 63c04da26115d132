"""bf16 prefill in tiles of 32, 64 and 128 rows (k_gemm_tile_short; run on an MI355X): every tile
height's edges, K split and not, X staged, read in place and rounded on the way."""

import numpy as np
import pytest

from oracle import mtc_oracle as O
from tensorpack_amd.core.allocation import rd_allocate
from tensorpack_amd.core.permutation import PermutedQuadtreeRD
from tensorpack_amd.core.quadtree import QuadtreeRD
from tensorpack_amd.kernels.gemm import MTCMatrix, mtc_gemm_group

from conftest import outlier_matrix

pytestmark = pytest.mark.gpu

# (K, N): a partial last K-step and column tile; one K-step; many K-steps (split K, several per block)
SHAPES = {"ragged": (992, 288), "one": (64, 256), "deep": (4096, 544)}


@pytest.fixture(scope="module")
def mats():
    out = {}
    for shape, (K, N) in SHAPES.items():
        W = outlier_matrix(K + N, K, N)
        h = np.exp(np.random.RandomState(K).randn(K))
        for form, bits in (("qt", 4.0), ("qtp", 3.5), ("p16", 11.0)):
            a = (PermutedQuadtreeRD if form == "qtp" else QuadtreeRD)(W, h, (32, 16, 8, 4)).select(bits)
            i = getattr(a, "inner", a)
            if form == "qtp":
                W_hat = O.permuted_qt_dequant(W, a.row_perm, a.col_perm, i.sizes, i.leaf, i.modes, i.scales)
            else:
                W_hat = O.qt_dequant(W, i.sizes, i.leaf, i.modes, i.scales)
            out[shape, form] = MTCMatrix.from_quadtree(a, W), W_hat
        al = rd_allocate(W, 4.5, None, 32)
        out[shape, "uniform"] = (MTCMatrix.from_allocation(W, al.modes, al.scales, 32),
                                 O.uniform_to_array(W, al.modes, al.scales, 32))
    return out


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
