"""What the planner chooses, on the CPU (tests/planner.py): every call over a range
of sizes, types, layouts and row strides is planned, its kernels are in the built
images, and each launch stays within what its kernel was built for."""

import itertools

import pytest

import kernel_isa as K
import planner

pytestmark = pytest.mark.skipif(not (K.tools_present() and K.images() and planner.buildable()),
                                reason="ROCm tools or built code objects absent")

LDS_PER_CU = 160 * 1024
NAME = {"f32": "float32", "f16": "float16", "bf16": "bfloat16"}
SIZE = {"f32": 4, "f16": 2, "bf16": 2}


@pytest.fixture(scope="module")
def limits():
    """kernel name -> (threads it may be launched with, bytes of its own LDS)."""
    return {name: (k[".max_flat_workgroup_size"], k[".group_segment_fixed_size"])
            for image in K.images() for name, k in K.metadata(image).items()}


def _check(limits, call):
    for name, grid, threads, lds in planner.launched():
        most, own = limits[name]
        assert threads <= most and own + lds <= LDS_PER_CU, (call, name, threads, lds)
        assert all(0 < g < 1 << 31 for g in grid), (call, name, grid)


def _matmul(element, layout, m, n, k, pad=0):
    """The launches of one product whose operands fill their buffers to the last
    element."""
    ops, Buffer = planner.package()
    lda = (m if layout == "tn" else k) + pad
    ldb = (k if layout == "nt" else n) + pad
    ldc = n + pad
    rows_a, rows_b = (k if layout == "tn" else m), (n if layout == "nt" else k)
    sizes = ((rows_a - 1) * lda + (lda - pad), (rows_b - 1) * ldb + (ldb - pad), m * ldc)
    buffers = [Buffer(s, NAME[element]) for s in sizes]
    strides = ((1, lda) if layout == "tn" else (lda, 1)) + \
        ((1, ldb) if layout == "nt" else (ldb, 1)) + (ldc, 1)
    try:
        ops.matmul(*buffers, m, n, k, strides=strides)
    finally:
        for b in buffers:
            b.free()


@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
@pytest.mark.parametrize("element", ["bf16", "f16", "f32"])
def test_products_are_planned(limits, element, layout):
    """Rows from a decoded token's to a batch's, columns from a tile's to a
    vocabulary's, 16-byte aligned rows (pad 0 or 8) and others."""
    planner.launched()
    for m, n, k, pad in itertools.product(
            (1, 2, 8, 16, 33, 64, 65, 200, 512, 1088, 2049), (1, 64, 200, 1000, 4096, 16640, 20000, 28672, 32000, 32128),
            (1, 32, 33, 64, 136, 770, 1024, 2048, 8192), (0, 8, 1)):
        _matmul(element, layout, m, n, k, pad)
        _check(limits, (element, layout, m, n, k, pad))


@pytest.mark.parametrize("layout,element,m,n,k", [
    ("nn", "bf16", 16, 28672, 8192), ("nn", "bf16", 16, 32000, 4096), ("nt", "f16", 32, 20000, 1024),
    ("tn", "bf16", 40, 32128, 2048), ("nn", "f16", 1, 16648, 8192),
])
def test_few_rows_of_many_columns_split_k(layout, element, m, n, k):
    """Decoding against a feed-forward or vocabulary projection: more 64 x 64 tiles
    than compute units, one wave group each, K in ranges across workgroups."""
    planner.launched()
    _matmul(element, layout, m, n, k)
    names = [x[0] for x in planner.launched()]
    suffix = "" if layout == "nn" else "_" + layout
    assert names == [f"tm_gemm_ragged{suffix}_t64_ks_{element}", f"tm_gemm_split_reduce_{element}"]


@pytest.mark.parametrize("element", ["bf16", "f16", "f32"])
def test_encoders_are_planned(limits, element):
    ops, Buffer = planner.package()
    planner.launched()
    encoder = ops.SAEEncoder(element)
    for m, d, f in itertools.product((1, 16, 65, 500, 2049, 8192), (1, 33, 64, 100, 768, 2048, 4097),
                                     (1, 64, 1000, 4096, 16384, 20000, 32001)):
        buffers = [Buffer(s, NAME[element]) for s in ((m, d), (d, f), (f,), (m, f))]
        encoder(*buffers)
        for b in buffers:
            b.free()
        _check(limits, (element, m, d, f))


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("element", ["bf16", "f16", "f32"])
def test_attention_is_planned(limits, element, causal):
    ops, _ = planner.package()
    planner.launched()
    for dim, heads, seq in itertools.product((1, 8, 20, 32, 40, 64, 72, 80, 96, 120, 127, 128), (1, 2, 7, 16, 40, 128),
                                             (1, 64, 129, 500, 1000, 1025, 2048, 4100)):
        layer = ops.AttentionLayer(heads, seq, dim, element, causal)
        layer.run_forward()
        layer.run_backward()
        layer.free()
        _check(limits, (element, causal, dim, heads, seq))
