"""The forms that small grids keep: the head_dim 64 dK/dV with one wave per SIMD and
fp32 attention on the fp32 MFMAs where the split form contracts columns that are not
there, against the fp64 oracle."""

import math

import pytest

from oracle import reference as R
from oracle import tolerance as T
from test_fast_paths_gpu import _attention, _check
from triton_metal import _core, ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("element", ["bf16", "f16"])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("heads,seq,pad", [
    (4, 1025, 0),  # one row in the last block
    (4, 1151, 8),
])
def test_dkdv_64_one_wave(device, element, causal, heads, seq, pad):
    out, variants, dense, _ = _attention(heads, seq, 64, element, causal, stride_seq=64 + pad)
    assert variants[3].endswith("_1w"), variants
    _check(out, dense, 64, causal, element=element)


@pytest.mark.parametrize("heads,seq", [(12, 1024), (29, 1100)])
def test_short_walks_and_larger_grids_take_two_waves(device, heads, seq):
    layer = ops.AttentionLayer(heads, seq, 64, "bf16")
    try:
        layer.run_forward()
        layer.run_backward()
        _core.synchronize()
        assert _core.kernel_variant(layer.lib.kernels["attn_bwd_dkdv"]) == "tm_attn_dkdv_fast_bf16_d64"
    finally:
        layer.free()


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("heads,seq,dim,pad,kept", [
    (2, 1, 80, 0, True), (3, 65, 65, 1, True), (6, 113, 80, 3, True), (2, 512, 72, 0, True),
    (2, 513, 80, 0, False), (2, 100, 81, 0, True), (65, 128, 80, 0, False),
])
def test_fp32_forward_65_to_80(device, heads, seq, dim, pad, causal, kept):
    out, variants, dense, _ = _attention(heads, seq, dim, "f32", causal, stride_seq=dim + pad)
    assert ("_mfma32" in variants[0]) == kept, variants
    want = R.attention_backward(*dense, 1 / math.sqrt(dim), causal)
    assert T.hybrid_error(out["o"], want["o"]) <= 2e-5
    assert T.hybrid_error(out["lse"], want["lse"]) <= 2e-5


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("heads,seq,dim,pad,kept", [
    # forward, dQ, dK/dV on the fp32 MFMAs
    (2, 97, 5, 2, "111"), (1, 1000, 20, 0, "111"), (6, 113, 40, 0, "111"),   # small, at most 40 columns
    (2, 97, 41, 1, "100"), (3, 65, 88, 0, "100"), (2, 96, 103, 1, "101"),    # the forward, dK/dV past 96
    (1, 129, 111, 1, "100"), (1, 129, 112, 0, "000"), (2, 96, 64, 0, "000"),
    (24, 300, 33, 0, "000"), (50, 150, 5, 2, "000"),                         # larger
    (24, 300, 72, 4, "100"), (24, 300, 81, 1, "000"), (24, 300, 100, 0, "001"), (24, 300, 104, 0, "000"), (24, 300, 96, 0, "000"),
])
def test_fp32_kernels_by_head_dimension(device, heads, seq, dim, pad, causal, kept):
    out, variants, dense, _ = _attention(heads, seq, dim, "f32", causal, stride_seq=dim + pad)
    names = (variants[0], variants[2], variants[3])
    assert "".join(str(int("_mfma32" in v)) for v in names) == kept, variants
    want = R.attention_backward(*dense, 1 / math.sqrt(dim), causal)
    assert T.hybrid_error(out["o"], want["o"]) <= 2e-5
    assert T.hybrid_error(out["lse"], want["lse"]) <= 2e-5
    for name in ("dq", "dk", "dv"):
        assert T.hybrid_error(out[name], want[name]) <= 1e-4, name
