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


@pytest.mark.parametrize("m,n,k,kernel,ranges", [
    (500, 500, 64, "generic", 1), (500, 500, 65, "x3_t64", 1), (2001, 2001, 64, "x3_t64", 1),
    (500, 500, 255, "x3_t64", 1), (500, 500, 256, "x3_t64", 2),       # 64 tiles
    (777, 777, 399, "x3_t64", 1), (777, 777, 400, "x3_t64", 3),       # 169
    (1001, 1001, 639, "x3_t64", 1), (1001, 1001, 640, "x3_t64", 4),   # 256
    (1001, 2003, 899, "x3_t64", 2), (1001, 2003, 900, "x3", 4),       # 128 tiles of 128 x 128
    (2001, 2001, 900, "x3", 2), (2001, 2050, 900, "x3_t64", 1),       # 256, 272
    (3001, 3001, 4000, "x3_t64", 1),                                  # 576
    (3585, 3457, 191, "x3_t64", 1), (3585, 3457, 192, "x3", 1),       # 812
    (2049, 3079, 1025, "x3", 1), (2305, 2400, 1000, "x3", 1), (2305, 2300, 1000, "x3_t64", 1),  # 425, 361, 342
    (16, 32001, 1000, "x3_t64", 2), (150, 20000, 1500, "x3_t64", 1),  # 128 x 128 tiles mostly empty
])
def test_fp32_tiles_and_ranges(m, n, k, kernel, ranges):
    """Each side of the lines between the fp32 GEMM's kernels (choose_gemm_x3,
    plan_x3_split), at sizes that fill no tile."""
    planner.launched()
    _matmul("f32", "nn", m, n, k, 1)
    launches = planner.launched()
    assert launches[0][0] == f"tm_gemm_{kernel}_f32"
    if kernel != "generic":
        assert launches[0][1][1] == ranges and len(launches) == (2 if ranges > 1 else 1)


def test_padded_forward_of_one_head(limits):
    """One long head of few columns: the generic forward in ranges, the padded
    backward; otherwise padded throughout from four workgroups on."""
    ops, _ = planner.package()
    for heads, seq, dim, forward, backward in (
            (1, 800, 32, "p32", "p32"), (1, 801, 32, "d32", "p32"), (1, 3000, 32, "d32", "p32"),
            (1, 3001, 32, "p32", "p32"), (2, 1000, 32, "p32", "p32"), (1, 1000, 56, "d64", "p64"),
            (1, 2049, 56, "p64", "p64"), (1, 1000, 72, "p80", "p80"), (1, 384, 80, "d96", "d96"),
            (1, 385, 80, "p80", "p80"), (4, 1, 80, "p80", "p80")):
        layer = ops.AttentionLayer(heads, seq, dim, "bf16")
        planner.launched()
        layer.run_forward()
        fwd = planner.launched()[0][0]
        layer.run_backward()
        bwd = [x[0] for x in planner.launched() if "_dq_" in x[0] or "_dkdv_" in x[0]]
        layer.free()
        assert fwd == f"tm_attn_fwd_generic_bf16_{forward}", (heads, seq, dim, fwd)
        assert len(bwd) == 2 and all(f"_generic_bf16_{backward}" in b for b in bwd), (heads, seq, dim, bwd)


@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
def test_wave_groups(limits, layout):
    """Waves a workgroup of the 16-bit 64 x 64 and 128 x 128 kernels has (two and four
    to a K group) on each side of the lines between one, two and four groups."""
    for m, n, k, groups in ((520, 520, 192, 1), (520, 520, 193, 2), (520, 520, 256, 2), (520, 520, 257, 4),
                            (1400, 1400, 255, 1), (1400, 1400, 256, 2),
                            (512, 512, 128, 4 if layout == "nn" else 1), (512, 512, 192, 4)):
        planner.launched()
        _matmul("bf16", layout, m, n, k, 8 if k % 8 == 0 else (-k) % 8 + 8)
        name, _, threads, _ = planner.launched()[0]
        assert threads == 128 * groups, (m, n, k, name, threads)
    for m, n, k, groups in ((2048, 2048, 128, 2 if layout == "nn" else 1), (2048, 2048, 192, 2),
                            (2304, 2176, 512, 2 if layout == "nn" else 1)):
        planner.launched()
        _matmul("bf16", layout, m, n, k)
        name, _, threads, _ = planner.launched()[0]
        assert "_t128" in name and threads == 256 * groups, (m, n, k, name, threads)
