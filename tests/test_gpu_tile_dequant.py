"""W_hat from the tile stream (mtc_tile_dequant, run on an MI355X): the oracle's bits for every cell
format, at shapes with partial K-steps and column tiles, several steps per block and negative scales."""

import numpy as np
import pytest

from oracle import mtc_oracle as O
from tensorpack_amd.core.allocation import rd_allocate
from tensorpack_amd.core.permutation import PermutedQuadtreeRD
from tensorpack_amd.core.quadtree import QuadtreeRD
from tensorpack_amd.device import DeviceTiles
from tensorpack_amd.kernels.gemm import MTCMatrix
from tensorpack_amd.packer import weight_codes
from tensorpack_amd.tilestream import pack_tiles

from conftest import outlier_matrix

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


@pytest.mark.parametrize("K,N,bits", [(32, 32, 6.0), (96, 288, 4.5), (1056, 544, 3.1), (4096, 3104, 2.6)])
@pytest.mark.parametrize("form", ["qt", "qtp", "qtp-scattered", "uniform"])
def test_tile_dequant_bit_exact(gpu, K, N, bits, form):
    W = outlier_matrix(K + N, K, N)
    h = np.exp(np.random.RandomState(K).randn(K))
    if form == "uniform":
        al = rd_allocate(W, bits, None, 32)
        # P0 blocks keep their +0.0 scale: from_allocation stores +0.0 for them whatever it is given, and
        # the oracle would multiply their zero codes by a -0.0
        flip = (np.random.RandomState(N).rand(*al.scales.shape) < 0.2) & (al.modes.reshape(al.scales.shape) > 0)
        scales = np.where(flip, -al.scales, al.scales).astype(np.float32)
        m = MTCMatrix.from_allocation(W, al.modes, scales, 32)
        want, tiles = O.uniform_to_array(W, al.modes, scales, 32), m.device_tiles(gpu)
    else:
        a = (QuadtreeRD if form == "qt" else PermutedQuadtreeRD)(W, h, (32, 16, 8, 4)).select(bits + 24.0 / min(K, N))
        i = getattr(a, "inner", a)
        if form == "qt":
            want, tiles = O.qt_dequant(W, i.sizes, i.leaf, i.modes, i.scales), MTCMatrix.from_quadtree(a, W).device_tiles(gpu)
        else:
            want = O.permuted_qt_dequant(W, a.row_perm, a.col_perm, i.sizes, i.leaf, i.modes, i.scales)
            tiles = DeviceTiles(pack_tiles((K, N), i.sizes, i.leaf, i.modes, i.scales,
                                           weight_codes(W[a.row_perm][:, a.col_perm]), "bf16", a.row_perm, a.col_perm,
                                           gather_cols=form == "qtp"), gpu)
    print("tile dequant", form, K, N, flush=True)
    assert np.array_equal(_bits(tiles.dequant().cpu().numpy()), _bits(want))


def test_dequant_device_takes_what_is_resident(gpu):
    """A matrix whose panel stream alone is on the device rebuilds W_hat from it; otherwise from tiles."""
    W = outlier_matrix(3, 256, 192)
    a = PermutedQuadtreeRD(W, None, (32, 16, 8, 4)).select(4.0)
    m, n = MTCMatrix.from_quadtree(a, W), MTCMatrix.from_quadtree(a, W)
    n.device_stream(None, gpu)
    got, panel = m.dequant_device(gpu), n.dequant_device(gpu)
    assert any(k[1] == "tiles" for k in m._dev) and not any(k[1] == "tiles" for k in n._dev)
    assert np.array_equal(_bits(got.cpu().numpy()), _bits(panel.cpu().numpy()))
