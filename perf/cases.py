"""Workloads of the packed-weight matmul, for timing and for comparing results.

Every case is one call through the public entry points: `mtc_gemm` (single matrix, fp32 decode /
fp32 results / bf16 prefill), `mtc_gemm_group` (matrices that read one input), the prepared batches
`GemvBatch` / `GemmBatch` (a decoder stack whose inputs are known together) and
`MTCMatrix.dequant_device` (the weight back in fp32). The offline allocator and the packers are not
timed: a program runs them once per weight, ahead of serving, on the CPU (they are part of `prepare`).

Weights. A real allocation of a 512 x 512 sample (the rate-distortion quadtree over the weight and
importance recipes of `tensorpack_amd.workloads`) gives a library of 256 root tiles with their
leaves, code widths and scales; a K x N matrix is laid out from these tiles (in sorted places for
permuted matrices, whose rows and columns are ordered by energy; anywhere otherwise). The weights
are exactly code * scale, so the quantizer finds the same codes again and `exact` needs only the
product. Uniform-block matrices draw a width per block and use the block's max-abs scale.

Case fields
  kind    gemm | group | gemv_batch | gemm_batch | dequant
  M, K, N rows of X, reduction rows, output columns (group / batches: K, N of the first matrix)
  form    qt | qtp (row/column-permuted) | uniform (one block size, fp32 scales)
  bits    allocator budget, bits per weight
  recipe  normal | student | blocks: weight distribution
  compute, x, y   mtc_gemm's compute, X dtype, Y dtype
  layers  decoder layers of a batch (7 matrices each)
"""

import math

import numpy as np
import torch

from tensorpack_amd.core.permutation import PermutedQTAllocation
from tensorpack_amd.core.quadtree import QTAllocation, QuadtreeRD
from tensorpack_amd.device import GemmBatch, GemvBatch
from tensorpack_amd.kernels.gemm import MTCMatrix, mtc_gemm, mtc_gemm_group
from tensorpack_amd.workloads import QWEN_LAYER

SAMPLE, ROOT, SIZES = 512, 32, (32, 16, 8, 4)
UNIQUE_LAYERS = 1        # layers of a stack packed apart; further layers are device copies of these
UNIFORM_MODES = ((0, 2, 3, 4, 5, 6, 8), (0.05, 0.15, 0.25, 0.30, 0.10, 0.05, 0.10))


def _case(kind, M, K, N, form="qt", bits=4.25, recipe="student", compute="auto", x="fp32", y="fp32", layers=0):
    return {"kind": kind, "M": M, "K": K, "N": N, "form": form, "bits": bits, "recipe": recipe, "compute": compute,
            "x": x, "y": y, "layers": layers}


def listed():
    cases = [
        # one small projection of a 0.5B decoder, one token: launch and latency bound
        ("decode 896x896 M1", _case("gemm", 1, 896, 896, "qtp", 3.125, "normal")),
        # one 4096-wide layer, one token: the decode headline
        ("decode 4096x4096 M1", _case("gemm", 1, 4096, 4096, "qtp", 4.25)),
        # a few sequences decoded together through a tall, narrow down projection (K split)
        ("decode 4864x896 M3", _case("gemm", 3, 4864, 896, "qtp", 3.125, "normal")),
        # sixteen sequences decoded together
        ("decode 4096x4096 M16", _case("gemm", 16, 4096, 4096, "qtp", 4.25)),
        # gate and up projections of one layer on the same token
        ("group gate+up M1", _case("group", 1, 896, 4864, "qtp", 3.125, "normal")),
        # a decoder stack's matrices for one token in one launch (8 layers, 56 matrices)
        ("stack decode M1", _case("gemv_batch", 1, 896, 896, "qtp", 3.125, "normal", layers=8)),
        # the same stack over a 512-token prompt
        ("stack prefill M512", _case("gemm_batch", 512, 896, 896, "qtp", 3.125, "normal", layers=8)),
        # a short prompt / a larger decode batch in bf16, ragged sizes, the uniform-block form
        ("prefill 2072x5472 M40", _case("gemm", 40, 2072, 5472, "uniform", 4.0, "normal", "auto", "bf16", "bf16")),
        # a 256-token prompt, block-scaled weights at few bits, fp32 activations
        ("prefill 4096x4096 M256", _case("gemm", 256, 4096, 4096, "qt", 2.5, "blocks")),
        # a long prompt through a large layer
        ("prefill 8192x8192 M4096", _case("gemm", 4096, 8192, 8192, "qt", 4.5, "student", "auto", "bf16")),
        # fp32 results above the decode sizes, an odd row count (evaluation, calibration)
        ("fp32 4096x4096 M100", _case("gemm", 100, 4096, 4096, "qtp", 4.25, "student", "fp32")),
        # the weight back in fp32 (export, checks, a cached dense copy)
        ("dequant 4096x4096", _case("dequant", 1, 4096, 4096, "qtp", 4.25)),
    ]
    return [dict(c, name=n) for n, c in cases]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ranges: any row count from one token to a 4096-row prompt, widths
    from 256 to 6144, every form, budgets of 2.5 to 5 bits, both compute paths and dtypes."""
    kind = rng.choice(["gemm"] * 10 + ["group", "group", "gemv_batch", "gemm_batch", "dequant"])
    K, N = 32 * _log(rng, 8, 192), 32 * _log(rng, 8, 192)
    form = rng.choice(["qt", "qtp", "qtp", "uniform"])
    bits = round(rng.uniform(2.5, 5.0), 2)
    recipe = rng.choice(["normal", "student", "student", "blocks"])
    if kind == "dequant":
        return _case(kind, 1, K, N, form, bits, recipe)
    if kind == "gemv_batch":
        return _case(kind, rng.choice([1, 1, 2, 4, 7, 12, 16]), 896, 896, "qtp", bits, recipe, layers=rng.randint(1, 8))
    if kind == "gemm_batch":
        return _case(kind, _log(rng, 17, 640), 896, 896, "qtp", bits, recipe, "auto", rng.choice(["fp32", "bf16"]),
                     layers=rng.randint(1, 6))
    if kind == "group":
        M = rng.choice([1, 2, 5, 16, _log(rng, 17, 512)])
        return _case(kind, M, min(K, 4096), N, form, bits, recipe)
    if form == "uniform":
        K += rng.choice([0, 8, 16, 24])
    path = rng.choice(["decode", "decode", "fp32", "bf16", "bf16"])
    if path == "decode":
        return _case(kind, rng.choice([1, 2, 3, 4, 5, 6, 8, 11, 16]), K, N, form, bits, recipe,
                     x=rng.choice(["fp32", "fp32", "bf16"]))
    if path == "fp32":
        return _case(kind, _log(rng, 17, 1024), K, N, form, bits, recipe, "fp32")
    return _case(kind, _log(rng, 17, 4096), K, N, form, bits, recipe, "auto", rng.choice(["bf16", "bf16", "fp32"]),
                 rng.choice(["fp32", "bf16"]))


# ---- weights ----
def _sample_weights(recipe, rng):
    n = SAMPLE
    if recipe == "blocks":
        W = rng.standard_normal((n, n)) * np.kron(10.0 ** rng.uniform(-3, 2, (n // ROOT, n // ROOT)), np.ones((ROOT, ROOT)))
        mask = rng.random((n, n)) < 0.02
        W = np.where(mask, np.where(rng.random((n, n)) < 0.5, 25.0, -25.0), W)
        return W.astype(np.float32), rng.lognormal(0.0, 1.0, n)
    W = (rng.standard_t(4, (n, n)) if recipe == "student" else rng.standard_normal((n, n))) * 0.02
    h = np.ones(n)
    h[rng.choice(n, n // 100, replace=False)] = 400.0        # outlier input channels, squared
    return W.astype(np.float32), h


def _expand(grid, s):
    return np.repeat(np.repeat(grid, s, axis=0), s, axis=1)


def _tiles(grid, per):
    """(g*per, g*per) grid -> (g*g, per, per), one entry per root tile."""
    g = grid.shape[0] // per
    return grid.reshape(g, per, g, per).swapaxes(1, 2).reshape(g * g, per, per)


def _quadtree(K, N, form, bits, recipe, rng):
    """(allocation, W_hat float32 in the original channel order) of a quadtree matrix."""
    W, h = _sample_weights(recipe, rng)
    permuted = form == "qtp"
    if permuted:
        e = h[:, None] * W.astype(np.float64) ** 2
        W = W[np.argsort(e.sum(axis=1), kind="stable")][:, np.argsort(e.sum(axis=0), kind="stable")]
        h = h[np.argsort(e.sum(axis=1), kind="stable")]
    a = QuadtreeRD(W, h, SIZES).select(bits)
    hat = np.zeros((SAMPLE, SAMPLE), np.float32)
    for s in SIZES:
        P, sc = _expand(np.where(a.leaf[s], a.modes[s], 0), s).astype(np.int64), _expand(a.scales[s], s)
        top = np.where(P > 0, 2.0 ** (np.maximum(P, 1) - 1), 0.0)
        q = np.clip(np.rint(W / np.where(P > 0, sc, 1.0)), -top, top - 1)
        hat += np.where(P > 0, q * sc, 0.0).astype(np.float32)     # 16 code bits x 8 scale bits: exact
    g, rk, rn = SAMPLE // ROOT, K // ROOT, N // ROOT
    if permuted:                                                   # sorted rows and columns: keep the place
        at = lambda n: np.clip(np.arange(n) * g // n + rng.integers(-1, 2, n), 0, g - 1)
        idx = at(rk)[:, None] * g + at(rn)[None, :]
    else:
        idx = rng.integers(0, g * g, (rk, rn))
    lay = lambda grid, s: np.ascontiguousarray(
        _tiles(grid, ROOT // s)[idx].swapaxes(1, 2).reshape(rk * (ROOT // s), rn * (ROOT // s)))
    leaf, modes, scales = ({s: lay(f[s], s) for s in SIZES} for f in (a.leaf, a.modes, a.scales))
    Wp = lay(hat, 1)
    inner = QTAllocation(SIZES, leaf, modes, scales, None, int(a.total_bits * (K * N) // SAMPLE ** 2), weights=Wp)
    if not permuted:
        return inner, Wp
    pr, pc = rng.permutation(K), rng.permutation(N)
    back = np.empty_like(Wp)
    back[np.ix_(pr, pc)] = Wp
    return PermutedQTAllocation(inner, pr, pc, inner.total_bits), back


def _uniform(K, N, recipe, rng):
    """(W, modes, scales, block size, W_hat in fp64) of a uniform-block matrix."""
    bs = next(b for b in (16, 8) if K % b == 0)
    W = rng.standard_normal((K, N), dtype=np.float32) * np.float32(0.02)
    if recipe == "blocks":
        W *= _expand((10.0 ** rng.uniform(-3, 2, (K // bs, N // bs))).astype(np.float32), bs)
    modes = rng.choice(UNIFORM_MODES[0], size=(K // bs, N // bs), p=UNIFORM_MODES[1]).astype(np.uint8)
    qmax = 2.0 ** (np.maximum(modes, 1).astype(np.float64) - 1) - 1
    peak = np.abs(W).reshape(K // bs, bs, N // bs, bs).max(axis=(1, 3))
    scales = (peak / np.maximum(qmax, 1.0)).astype(np.float32)
    P, sc = _expand(modes, bs), _expand(scales, bs)
    top = np.where(P > 0, 2.0 ** (np.maximum(P, 1).astype(np.int64) - 1), 0.0)
    q = np.clip(np.rint(W / sc), -top, np.maximum(top - 1, 0.0))
    return W, modes, scales, bs, np.where(P > 0, q * sc.astype(np.float64), 0.0)


def _matrix(K, N, case, rng):
    """(MTCMatrix, W_hat as a numpy array in the original channel order)."""
    if case["form"] == "uniform":
        W, modes, scales, bs, hat = _uniform(K, N, case["recipe"], rng)
        return MTCMatrix.from_allocation(W, modes, scales, bs), hat
    alloc, hat = _quadtree(K, N, case["form"], case["bits"], case["recipe"], rng)
    return MTCMatrix.from_quadtree(alloc), hat


def _shapes(case):
    if case["kind"] in ("gemv_batch", "gemm_batch"):
        return [(K, N) for _ in range(case["layers"]) for _, K, N in QWEN_LAYER]
    if case["kind"] == "group":
        return [(case["K"], case["N"])] * 2
    return [(case["K"], case["N"])]


def _activations(case, seed, device):
    """The inputs, one per matrix of a batch, else one: normal activations with 1 % outlier channels."""
    g = torch.Generator(device="cpu").manual_seed(int(seed) * 2 + 1)
    shapes = _shapes(case)
    if case["kind"] not in ("gemv_batch", "gemm_batch"):
        shapes = shapes[:1]
    out = []
    for K, _ in shapes:
        scale = torch.where(torch.rand(K, generator=g) < 0.01, 20.0, 1.0)
        X = torch.randn(case["M"], K, generator=g) * scale
        out.append(X.to(device=device, dtype=torch.bfloat16 if case["x"] == "bf16" else torch.float32))
    return out


def _weights(case, seed):
    """The distinct (MTCMatrix, W_hat) of a case and, per matrix of the call, which of them it is."""
    rng = np.random.default_rng(int(seed))
    shapes = _shapes(case)
    n = min(len(shapes), UNIQUE_LAYERS * len(QWEN_LAYER)) if case["layers"] else len(shapes)
    return [_matrix(K, N, case, rng) for K, N in shapes[:n]], [i % n for i in range(len(shapes))]


def prepare(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    mats, which = _weights(case, seed)
    mats = [m for m, _ in mats]
    Xs = _activations(case, seed, dev)
    state = {"case": case, "mats": mats, "Xs": Xs}
    if case["kind"] == "gemv_batch":
        streams = [m.device_stream(M=case["M"]) for m in mats]
        state["batch"] = GemvBatch([streams[w] if i < len(mats) else streams[w].clone() for i, w in enumerate(which)], Xs)
    elif case["kind"] == "gemm_batch":
        tiles = [m.device_tiles() for m in mats]
        state["batch"] = GemmBatch([tiles[w] if i < len(mats) else tiles[w].clone() for i, w in enumerate(which)], Xs)
    else:
        # a program's warm-up call at its own size: the layouts this call needs are then on the GPU
        run({**state, "Xs": [torch.zeros_like(x) for x in Xs]})
    for m in mats:
        m.release_host_streams()
    return state


_DTYPE = {"fp32": torch.float32, "bf16": torch.bfloat16}


def run(state):
    case = state["case"]
    if case["kind"] in ("gemv_batch", "gemm_batch"):
        return state["batch"].launch()
    if case["kind"] == "dequant":
        return state["mats"][0].dequant_device()
    if case["kind"] == "group":
        return mtc_gemm_group(state["Xs"][0], state["mats"], compute=case["compute"])
    return mtc_gemm(state["Xs"][0], state["mats"][0], compute=case["compute"], out_dtype=_DTYPE[case["y"]])


def work(case):
    M, xb, yb = case["M"], 2 if case["x"] == "bf16" else 4, 2 if case["y"] == "bf16" else 4
    shapes = _shapes(case)
    weights = sum(K * N for K, N in shapes)
    packed = weights * case["bits"] / 8
    if case["kind"] == "dequant":
        return {"bytes": packed + 4 * weights, "flops": weights}
    xs = shapes if case["kind"] in ("gemv_batch", "gemm_batch") else shapes[:1]
    return {"bytes": packed + xb * M * sum(K for K, _ in xs) + yb * M * sum(N for _, N in shapes),
            "flops": 2 * M * weights}


def tolerance(case):
    if case["kind"] == "dequant":
        return "exact" if case["form"] != "uniform" else {"rel": 1e-7, "max": 2e-7}   # one fp32 product per weight
    if case["compute"] == "fp32" or (case["M"] <= 16 and case["kind"] != "gemm_batch"):
        return {"rel": 2e-6, "max": 2e-5}     # fp32 products and sums (against `exact`: up to 5.7e-7, 4.6e-6)
    return {"rel": 1e-2, "max": 0.1}          # operands (and results, where asked) rounded to bf16: 2.8e-3, 2.5e-2


def exact(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    mats, which = _weights(case, seed)
    hats = [torch.from_numpy(np.ascontiguousarray(h)).to(dev).double() for _, h in mats]
    if case["kind"] == "dequant":
        return hats[0]
    Xs = [x.double() for x in _activations(case, seed, dev)]
    if case["kind"] in ("gemv_batch", "gemm_batch"):
        return [x @ hats[w] for x, w in zip(Xs, which)]
    if case["kind"] == "group":
        return [Xs[0] @ h for h in hats]
    return Xs[0] @ hats[0]
