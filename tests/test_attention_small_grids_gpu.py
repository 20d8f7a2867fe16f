"""The forms that small grids keep: the head_dim 64 dK/dV with one wave per SIMD, against the fp64 oracle."""

import pytest

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
