"""fp32 GEMM and SAE encoder on the bf16 matrix cores (three-way split): every
layout and tile size, ragged and odd shapes, K ranges, against fp64 within the
fp32 accumulation bound K 2^-24 (|A| |B|), which also holds for the smallest values
there are and for values and results past the range of the split (the fp32
fallback); sums of few products within their last places."""

import numpy as np
import pytest

from oracle import reference as R
from triton_metal import _core, ops
from triton_metal.buffer import DeviceBuffer

pytestmark = pytest.mark.gpu


def _run(a, b, layout, pad):
    """C, the variant, for A [m, k] and B [k, n] stored with `pad` elements of
    inf behind every row; C is fenced with -7."""
    (m, k), n = a.shape, b.shape[1]
    def stored(x):
        y = np.full((x.shape[0], x.shape[1] + pad), np.inf, np.float32)
        y[:, :x.shape[1]] = x
        return y
    sa, sb = stored(a.T if layout == "tn" else a), stored(b.T if layout == "nt" else b)
    lda, ldb = sa.shape[1], sb.shape[1]
    strides = ((1, lda) if layout == "tn" else (lda, 1)) + ((1, ldb) if layout == "nt" else (ldb, 1)) + (n + pad, 1)
    A, B = DeviceBuffer.from_numpy(sa), DeviceBuffer.from_numpy(sb)
    C = DeviceBuffer.from_numpy(np.full((m + 2, n + pad), -7.0, np.float32))
    try:
        ops.matmul(A, B, C, m, n, k, strides=strides)
        variant = _core.kernel_variant(ops.library("f32").kernels["matmul_kernel"])
        c = C.numpy()
    finally:
        for x in (A, B, C):
            x.free()
    assert np.all(c[:, n:] == -7.0) and np.all(c[m:] == -7.0)
    return c[:m, :n], variant


def _check(c, a, b, k):
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    bound = max(k, 32) * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64)) + 2.0 ** -149 * k
    assert np.all(np.abs(c - a64 @ b64) <= bound)


@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
@pytest.mark.parametrize("m,n,k,pad,kernel", [
    (1, 1, 33, 1, "generic"),          # few tiles of two steps
    (65, 63, 64, 1, "generic"),
    (1, 1, 65, 1, "_t64"),
    (65, 63, 96, 1, "_t64"),           # whole steps
    (129, 257, 65, 3, "_t64"),
    (64, 200, 1000, 2, "_t64"),        # K ranges
    (1409, 1281, 161, 1, "_t64"),      # 23 x 21 tiles
    (1409, 1281, 993, 1, ""),          # 12 x 11 tiles of 128, K ranges
    (2177, 2050, 95, 1, "_t64"),       # 35 x 33 tiles
    (3585, 3457, 259, 1, ""),          # 29 x 28 tiles of 128
    (2304, 2176, 64, 0, "_t64"),       # whole tiles, more than one per compute unit
    (3584, 3584, 256, 0, ""),          # and three of 128 x 128
    (2048, 1024, 1056, 0, ""),         # whole 128 x 128 tiles for half of them, long K
    (128, 320, 512, 0, "_t64"),        # whole 64 x 64 tiles, few
    (1088, 1024, 768, 0, "_t64"),      # and more than one per compute unit
])
def test_x3_gemm(device, layout, m, n, k, pad, kernel):
    rng = np.random.default_rng(m + n + k)
    a = rng.standard_normal((m, k), dtype=np.float32)
    b = rng.standard_normal((k, n), dtype=np.float32)
    c, got = _run(a, b, layout, pad)
    suffix = "" if layout == "nn" else "_" + layout
    assert got.split(" + ")[0] == ("tm_gemm_generic_f32" if kernel == "generic" else f"tm_gemm_x3{suffix}{kernel}_f32")
    _check(c, a, b, k)


@pytest.mark.parametrize("m,n,k,layout", [(2048, 1088, 8192, "nn"), (1088, 2048, 8192, "tn")])
def test_x3_operands_of_whole_2_mib(device, m, n, k, layout):
    """128 x 128 tiles, the last one 64 wide, over an operand that ends where its
    allocation ends (tests/test_x3_runs.py: no load leaves it)."""
    rng = np.random.default_rng(4)
    a = rng.standard_normal((m, k), dtype=np.float32)
    b = rng.standard_normal((k, n), dtype=np.float32)
    c, got = _run(a, b, layout, 0)
    assert got.split(" + ")[0] == f"tm_gemm_x3{'_tn' if layout == 'tn' else ''}_f32"
    _check(c, a, b, k)


@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
@pytest.mark.parametrize("scale", [2.0 ** -115, 2.0 ** -99, 2.0 ** 60, 2.0 ** 100])
def test_x3_keeps_small_and_large_values(device, layout, scale):
    """A near the bottom of the range (its low parts subnormal but for the factor the
    split gives them) and near the top, B such that the products stay in range."""
    rng = np.random.default_rng(2)
    m, n, k = 70, 90, 77
    a = (rng.standard_normal((m, k)) * scale).astype(np.float32)
    b = (rng.standard_normal((k, n)) / scale).astype(np.float32)
    c, got = _run(a, b, layout, 1)
    assert "_x3" in got
    _check(c, a, b, k)


def test_x3_values_that_round_past_bf16(device):
    """3.4e38 rounds to infinity in bf16: the tile is computed in fp32."""
    m, n, k = 40, 40, 70
    a = np.full((m, k), np.float32(3.4e38))
    b = np.zeros((k, n), np.float32)
    b[3] = 0.5
    c, got = _run(a, b, "nn", 1)
    assert "_x3" in got
    assert np.all(c == np.float32(1.7e38))


def test_x3_infinities_and_nan(device):
    """As fp32 arithmetic has them: inf times a number, inf - inf, NaN, and no
    trace in the rows that hold none."""
    rng = np.random.default_rng(2)
    m, n, k = 70, 66, 82
    a = rng.standard_normal((m, k), dtype=np.float32)
    b = np.abs(rng.standard_normal((k, n), dtype=np.float32)) + 0.5
    a[0, 3] = np.inf
    a[1, 4] = -np.inf
    a[2, 5], a[2, 6] = np.inf, -np.inf
    a[69, 81] = np.nan
    c, got = _run(a, b, "nn", 1)
    assert "_x3" in got
    assert np.all(c[0] == np.inf) and np.all(c[1] == -np.inf)
    assert np.all(np.isnan(c[2])) and np.all(np.isnan(c[69]))
    rows = [i for i in range(m) if i not in (0, 1, 2, 69)]
    _check(c[rows], a[rows], b, k)


def test_x3_whole_numbers_are_exact(device):
    rng = np.random.default_rng(2)
    a = rng.integers(-500, 500, (130, 200)).astype(np.float32)
    b = rng.integers(-50, 50, (200, 70)).astype(np.float32)
    c, got = _run(a, b, "nn", 1)
    assert "_x3" in got
    assert np.array_equal(c, (a.astype(np.float64) @ b).astype(np.float32))


@pytest.mark.parametrize("rows,model,features", [(33, 65, 129), (24, 900, 700), (2305, 70, 2200), (2304, 64, 2304)])
def test_x3_sae(device, rows, model, features):
    rng = np.random.default_rng(5)
    x = rng.standard_normal((rows, model), dtype=np.float32)
    w = rng.standard_normal((model, features), dtype=np.float32) / np.float32(np.sqrt(model))
    b = rng.standard_normal(features, dtype=np.float32)
    enc = ops.SAEEncoder("f32")
    got = enc.numpy(x, w, b)
    assert "_x3" in _core.kernel_variant(enc.kernel)
    want = R.sae_encode(x, w, b)
    bound = (model + 1) * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(w) + np.abs(b))
    assert np.all(np.abs(got - want) <= bound)


@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
def test_x3_keeps_subnormal_values_and_results(device, layout):
    """Every fp32 number is split without loss, beside ordinary ones; results are
    rounded once more where fp32 itself is short of bits."""
    rng = np.random.default_rng(3)
    m, n, k = 70, 90, 77
    a = rng.standard_normal((m, k)).astype(np.float32)
    b = rng.standard_normal((k, n)).astype(np.float32)
    a[:20] = np.ldexp(a[:20], -135)
    b[:, :30] = np.ldexp(b[:, :30], 100)
    c, got = _run(a, b, layout, 1)
    assert "_x3" in got
    _check(c, a, b, k)


@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
@pytest.mark.parametrize("m,n,k,power", [(140, 130, 65, 40), (140, 130, 65, 55), (1409, 1281, 77, 50), (64, 200, 1000, 50)])
def test_x3_results_past_the_scaled_range(device, layout, m, n, k, power):
    """Results from 2^96 on are computed in fp32: both tile sizes, K ranges."""
    rng = np.random.default_rng(4)
    a = np.ldexp(rng.standard_normal((m, k)), power).astype(np.float32)
    b = np.ldexp(rng.standard_normal((k, n)), power).astype(np.float32)
    b[:, 64:] = np.ldexp(b[:, 64:], -power)
    c, got = _run(a, b, layout, 1)
    assert "_x3" in got
    _check(c, a, b, k)


@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
@pytest.mark.parametrize("m,n,k", [(257, 259, 1025), (1409, 1281, 993)])
@pytest.mark.parametrize("terms", [1, 2, 4])
def test_x3_sums_of_few_products(device, layout, m, n, k, terms):
    """Full-width values, one product to a 32-wide step and `terms` in all: a lone
    product is within 0.52 of its last place (0.5, and what the seven small partial
    products, 2^-8 of it, are rounded by), and each further one adds an accumulation
    of the 16-bit MFMA, whose single steps are up to 0.875 off."""
    rng = np.random.default_rng(terms)
    full = lambda *shape: (rng.uniform(1, 2, shape) * np.exp2(rng.integers(-8, 8, shape)) *
                           rng.choice((-1, 1), shape)).astype(np.float32)
    a, b = np.zeros((m, k), np.float32), full(k, n)
    for t in range(terms):
        a[np.arange(m), (np.arange(m) * 7 + t * (k // terms)) % k] = full(m)
    c, got = _run(a, b, layout, 1)
    assert "_x3" in got
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    ulp = np.exp2(np.floor(np.log2(np.abs(a64) @ np.abs(b64))) - 23)
    assert np.max(np.abs(c - a64 @ b64) / ulp) <= 0.52 + 0.875 * (terms - 1)
