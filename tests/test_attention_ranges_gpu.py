"""The 16-bit dQ and dK/dV kernels over ranges of their walk (few heads, long
sequences) against the fp64 oracle, padded rows and ragged ends included."""

import pytest

from test_fast_paths_gpu import _attention, _check
from triton_metal import _core, ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("element", ["bf16", "f16"])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("heads,seq,dim,pad", [
    (1, 768, 64, 0),       # three ranges of four 64-key blocks
    (3, 1001, 64, 8),      # a ragged last block
    (1, 1000, 128, 0),
    (2, 833, 80, 8), (2, 1025, 32, 0), (1, 800, 96, 0), (1, 900, 112, 0),
])
def test_backward_ranges(device, element, causal, heads, seq, dim, pad):
    out, variants, dense, _ = _attention(heads, seq, dim, element, causal, stride_seq=dim + pad)
    assert all("_ranges + tm_attn_split_reduce_" in v for v in variants[2:]), variants
    _check(out, dense, dim, causal, element=element)


def test_short_walks_and_many_heads_keep_the_whole_walk(device):
    for heads, seq in ((1, 767), (40, 768)):
        layer = ops.AttentionLayer(heads, seq, 64, "bf16")
        try:
            layer.run_forward()
            layer.run_backward()
            _core.synchronize()
            for name in ("attn_bwd_dq", "attn_bwd_dkdv"):
                assert "ranges" not in _core.kernel_variant(layer.lib.kernels[name])
        finally:
            layer.free()
