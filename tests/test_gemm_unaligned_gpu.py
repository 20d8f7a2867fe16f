"""16-bit GEMMs and SAE encoders whose rows start at any 2-byte address, against
fp64: every layout, tile size and K split, with inf and NaN in the operands'
padding and sentinels around C."""

import numpy as np
import pytest

from oracle import reference as R
from oracle import tolerance as T
from test_fast_paths_gpu import _gemm, _gemm_nt, _gemm_tn
from triton_metal import _core, ops
from triton_metal.buffer import round_to

pytestmark = pytest.mark.gpu

SHAPES = [
    (1, 1, 1, "generic"),             # one element
    (3, 5, 7, "generic"),
    (64, 64, 64, "generic"),          # one whole tile and step
    (65, 63, 65, "generic"),          # one past and one short
    (129, 257, 127, "generic"),
    (100, 90, 1001, "unaligned_t64_ks"),     # K ranges, a ragged last step
    (2049, 2111, 63, "unaligned_t128"),      # shorter than one step
    (2305, 2049, 129, "unaligned_t128"),
    (4097, 4103, 65, "unaligned"),           # 256 x 256 tiles, one past whole
    (3841, 4095, 128, "unaligned"),          # whole steps
]


@pytest.mark.parametrize("element", ["bf16", "f16"])
@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
@pytest.mark.parametrize("m,n,k,kernel", SHAPES)
def test_unaligned_gemm(device, element, layout, m, n, k, kernel):
    # odd leading dimensions past the matrix, so padding lies behind every row
    odd = lambda x: x + 1 + (x % 2)
    if layout == "nn":
        c, want, got = _gemm(m, n, k, element, odd(k), odd(n), odd(n), poison=True, extra_rows=3)
    elif layout == "nt":
        c, want, got = _gemm_nt(m, n, k, element, odd(k), odd(k), odd(n))
    else:
        c, want, got = _gemm_tn(m, n, k, element, odd(m), odd(n), odd(n))
        kernel = "unaligned_t128" if kernel == "unaligned" else kernel
    if kernel != "generic" and layout != "nn":
        kernel = kernel.replace("unaligned", "unaligned_" + layout)
    assert got.split(" + ")[0] == f"tm_gemm_{kernel}_{element}"
    assert np.all(np.isfinite(c[:m, :n]))
    assert T.hybrid_error(c[:m, :n], want) <= 2e-2
    assert np.all(c[:m, n:] == -7.0) and np.all(c[m:] == -7.0)


@pytest.mark.parametrize("element", ["bf16", "f16"])
@pytest.mark.parametrize("k", [64, 70])
def test_rows_of_c_at_any_address(device, element, k):
    """Aligned operands with an odd row stride of C keep the aligned copies."""
    c, want, got = _gemm(192, 256, k, element, 72, 256, 257, extra_rows=3)
    assert got == f"tm_gemm_ragged_t64_{element}"
    assert T.hybrid_error(c[:192, :256], want) <= 2e-2
    assert np.all(c[:192, 256:] == -7.0) and np.all(c[192:] == -7.0)


@pytest.mark.parametrize("strided", ["both", "k"])
def test_strides_that_are_not_unit(device, strided):
    """Strides of 2 in both dimensions of A (or along K only) take the fp32-MFMA
    body of the generic kernel."""
    from triton_metal.buffer import DeviceBuffer
    m, n, k = 70, 50, 33
    rng = np.random.default_rng(3)
    a = round_to(rng.standard_normal((2 * m, 2 * k), dtype=np.float32), "bf16")
    b = round_to(rng.standard_normal((k, n), dtype=np.float32), "bf16")
    A, B, C = DeviceBuffer.from_numpy(a, "bfloat16"), DeviceBuffer.from_numpy(b, "bfloat16"), \
        DeviceBuffer((m, n), "bfloat16")
    sam = 4 * k if strided == "both" else 2 * k
    try:
        ops.matmul(A, B, C, m, n, k, strides=(sam, 2, n, 1, n, 1))
        assert _core.kernel_variant(ops.library("bf16").kernels["matmul_kernel"]) == "tm_gemm_generic_bf16"
        c = C.float32()
    finally:
        for x in (A, B, C):
            x.free()
    rows = a[::2] if strided == "both" else a[:m]
    want = rows[:m, ::2].astype(np.float64) @ b.astype(np.float64)
    assert T.hybrid_error(c, want) <= 2e-2


@pytest.mark.parametrize("element", ["bf16", "f16"])
@pytest.mark.parametrize("rows,model,features,kernel", [
    (33, 65, 129, "generic"), (2049, 63, 2111, "unaligned_t128"), (4097, 65, 4103, "unaligned")])
def test_unaligned_sae(device, element, rows, model, features, kernel):
    rng = np.random.default_rng(5)
    x = round_to(rng.standard_normal((rows, model), dtype=np.float32), element)
    w = round_to(rng.standard_normal((model, features), dtype=np.float32) / np.sqrt(model), element)
    b = round_to(rng.standard_normal(features, dtype=np.float32), element)
    enc = ops.SAEEncoder(element)
    got = enc.numpy(x, w, b)
    assert _core.kernel_variant(enc.kernel) == f"tm_sae_{kernel}_{element}"
    assert T.hybrid_error(got, R.sae_encode(x, w, b)) <= 2e-2


@pytest.mark.parametrize("m,k", [(2048, 1025), (1 << 20, 1)])
def test_operand_that_ends_its_allocation(device, m, k):
    """A fills its buffer.  At 2^20 x 1 that is whole 2 MiB, allocated as asked
    with nothing behind it, so the loads that reach past the end are not taken;
    elsewhere the allocation has room for them."""
    from triton_metal.buffer import DeviceBuffer
    n = 3
    rng = np.random.default_rng(3)
    a = round_to(rng.standard_normal((m, k), dtype=np.float32), "bf16")
    b = round_to(rng.standard_normal((k, n), dtype=np.float32), "bf16")
    A, B, C = DeviceBuffer.from_numpy(a, "bfloat16"), DeviceBuffer.from_numpy(b, "bfloat16"), \
        DeviceBuffer((m, n), "bfloat16")
    try:
        ops.matmul(A, B, C, m, n, k)
        c = C.float32()
    finally:
        for x in (A, B, C):
            x.free()
    assert T.hybrid_error(c, a.astype(np.float64) @ b.astype(np.float64)) <= 2e-2
