"""16-bit attention at head dimensions other than 64 and 128: the padded MFMA
kernels (tm_attn_*_generic_<type>_p<width>), forward and backward against the
fp64 oracle at the edges of their tiles, with the rows' padding poisoned."""

import math

import numpy as np
import pytest

from oracle import reference as R
from oracle import tolerance as T
from triton_metal import _core, ops
from triton_metal.buffer import DeviceBuffer, round_to

pytestmark = pytest.mark.gpu

DT = {"f16": "float16", "bf16": "bfloat16"}
WIDTHS = (32, 64, 80, 96, 128)


def _run(heads, seq, dim, element, causal, pad, seed):
    """Rows of dim + pad elements whose padding holds inf in the operands and
    5 in the outputs; returns outputs, whole output rows and variants."""
    ss = dim + pad
    rng = np.random.default_rng(seed)
    dense = [round_to(rng.standard_normal((heads, seq, dim), dtype=np.float32), element)
             for _ in range(4)]
    rows = np.full((heads, seq, ss), np.inf, np.float32)
    bufs = {}
    for name, x in zip(("q", "k", "v", "do"), dense):
        rows[:, :, :dim] = x
        bufs[name] = DeviceBuffer.from_numpy(rows, DT[element])
    for name in ("o", "dq", "dk", "dv"):
        bufs[name] = DeviceBuffer.from_numpy(np.full((heads, seq, ss), 5.0, np.float32), DT[element])
    for name in ("lse", "delta"):
        bufs[name] = DeviceBuffer((heads, seq), "float32")
    kern = ops.library(element, dim, causal).kernels
    h = lambda names: [bufs[n].tm_handle for n in names.split()]
    B, I, F = _core.ARG_BUFFER, _core.ARG_I32, _core.ARG_F32
    scale = _core.float_bits(1 / math.sqrt(dim))
    variants = []
    try:
        for name, kinds, values in (
                ("attn_fwd", [B] * 4 + [F, I, I, I, B, I],
                 h("q k v o") + [scale, seq * ss, ss, seq] + h("lse") + [seq]),
                ("attn_bwd_preprocess", [B] * 3 + [I] * 4, h("o do delta") + [seq * ss, ss, seq, seq]),
                ("attn_bwd_dq", [B] * 7 + [F] + [I] * 4,
                 h("q k v do dq lse delta") + [scale, seq * ss, ss, seq, seq]),
                ("attn_bwd_dkdv", [B] * 8 + [F] + [I] * 4,
                 h("q k v do dk dv lse delta") + [scale, seq * ss, ss, seq, seq])):
            _core.launch(kern[name], (1, heads, 1), 128, kinds, values)
            variants.append(_core.kernel_variant(kern[name]))
        out = {n: bufs[n].float32() for n in ("o", "lse", "dq", "dk", "dv")}
    finally:
        for b in bufs.values():
            b.free()
    return dense, out, variants


@pytest.mark.parametrize("element", ["bf16", "f16"])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("seq", [1, 64, 129, 300])
@pytest.mark.parametrize("dim,pad", [(8, 8), (32, 0), (40, 8), (72, 8), (80, 0), (88, 16), (96, 0),
                                     (120, 8), (104, 0)])
def test_padded_head_dims(device, element, causal, seq, dim, pad):
    """Every tolerance is that of the other 16-bit kernels, except L, whose row
    sums are fp32 sums of the unrounded P: the fp32 tests' 2e-5."""
    heads = 5
    dense, out, variants = _run(heads, seq, dim, element, causal, pad, seed=seq * 131 + dim)
    width = next(w for w in WIDTHS if dim <= w)
    want_variant = f"_generic_{element}_p{width}" + ("_causal" if causal else "")
    assert all(want_variant in v for i, v in enumerate(variants) if i != 1), variants
    want = R.attention_backward(*dense, 1 / math.sqrt(dim), causal)
    tol = 2e-2 if element == "bf16" else 4e-3
    assert T.max_abs_error(out["o"][:, :, :dim], want["o"]) <= tol
    assert T.hybrid_error(out["lse"], want["lse"]) <= 2e-5
    for name in ("dq", "dk", "dv"):
        assert T.hybrid_error(out[name][:, :, :dim], want[name]) <= tol, name
    for name in ("o", "dq", "dk", "dv"):
        assert np.all(out[name][:, :, dim:] == 5.0), name


def test_offsets_move_when_scores_grow(device):
    """Scores that rise along the keys by more than the exponent bias of P move
    the row offsets in later blocks; the row sums kept beside the exponentials
    are taken back and scaled with them."""
    heads, seq, dim = 4, 400, 80
    rng = np.random.default_rng(4)
    q = round_to(rng.standard_normal((heads, seq, dim), dtype=np.float32), "f16")
    k = round_to(rng.standard_normal((heads, seq, dim), dtype=np.float32)
                 * (1 + np.arange(seq, dtype=np.float32) / 40)[None, :, None], "f16")
    v = round_to(rng.standard_normal((heads, seq, dim), dtype=np.float32), "f16")
    layer = ops.AttentionLayer(heads, seq, dim, "f16")
    try:
        o, lse = layer.forward(q, k, v)
        assert "_p80" in _core.kernel_variant(layer.lib.kernels["attn_fwd"])
    finally:
        layer.free()
    want_o, _, want_l = R.attention_forward(q, k, v, 1 / math.sqrt(dim), False)
    assert T.max_abs_error(o, want_o) <= 4e-3
    assert T.hybrid_error(lse, want_l) <= 2e-5


@pytest.mark.parametrize("dim", [32, 80, 120])
def test_small_probabilities_keep_their_bits(device, dim):
    """f16 holds P unscaled: 89 x 2^-24, a value of f16, for every key but the first,
    which holds the row maximum and a V of 0."""
    heads, seq = 4, 512
    q, k = (np.zeros((heads, seq, dim), np.float32) for _ in range(2))
    q[:, :, 0] = 1.0
    k[:, 1:, 0] = -1.0
    v = np.ones((heads, seq, dim), np.float32)
    v[:, 0] = 0.0
    layer = ops.AttentionLayer(heads, seq, dim, "f16", scale=math.log(2.0 ** 24 / 89))
    try:
        o, _ = layer.forward(q, k, v)
        assert "_generic_f16_p" in _core.kernel_variant(layer.lib.kernels["attn_fwd"])
    finally:
        layer.free()
    p = 89 * 2.0 ** -24
    want = (seq - 1) * p / (1 + (seq - 1) * p)
    assert np.max(np.abs(o - want)) <= 2e-3 * want  # the rounding of O is 2^-11, a bias of 2^-2 11e-3
