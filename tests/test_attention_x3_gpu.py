"""fp32 attention on the bf16 matrix cores (three-way split operands): block and
head-dimension edges, odd strides, the smallest values, probabilities and score
gradients, and values and scores past the range of the split, which the generic body
computes, all at the fp32 tests' bounds.  (Small grids of head dimensions that are
no multiple of 32 run the fp32 MFMAs: test_attention_small_grids_gpu.py has larger
ones.)"""

import math

import numpy as np
import pytest

from oracle import reference as R
from oracle import tolerance as T
from test_fast_paths_gpu import _attention
from triton_metal import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("heads,seq,dim,pad", [
    (2, 1, 64, 0), (2, 63, 64, 1), (3, 65, 64, 3), (1, 130, 33, 0), (2, 97, 5, 2), (2, 31, 96, 1),
    (1, 33, 127, 0), (9, 200, 128, 4), (40, 520, 64, 0), (70, 130, 32, 0),
])
def test_edges(device, heads, seq, dim, pad, causal):
    """Head dimensions that are no multiple of 8, rows at any 4-byte address,
    split (few heads) and whole walks."""
    out, variants, dense, _ = _attention(heads, seq, dim, "f32", causal, stride_seq=dim + pad)
    assert "_generic_f32_d" in variants[0]
    want = R.attention_backward(*dense, 1 / math.sqrt(dim), causal)
    assert T.hybrid_error(out["o"], want["o"]) <= 2e-5
    assert T.hybrid_error(out["lse"], want["lse"]) <= 2e-5
    for name in ("dq", "dk", "dv"):
        assert T.hybrid_error(out[name], want[name]) <= 1e-4, name


def _layer(x, scale, causal=False):
    heads, seq, dim = x["q"].shape
    layer = ops.AttentionLayer(heads, seq, dim, "f32", causal, scale=scale)
    try:
        o, lse = layer.forward(x["q"], x["k"], x["v"])
        dq, dk, dv = layer.backward(x["do"])
    finally:
        layer.free()
    return {"o": o, "lse": lse, "dq": dq, "dk": dk, "dv": dv}


def _inputs(heads=2, seq=150, dim=64, seed=3):
    rng = np.random.default_rng(seed)
    return {n: rng.standard_normal((heads, seq, dim), dtype=np.float32) for n in ("q", "k", "v", "do")}


@pytest.mark.parametrize("name,power", [("k", -110), ("q", -115), ("v", -105), ("do", -108)])
def test_values_below_the_split(device, name, power):
    """One tensor near the bottom of the range: gradients and outputs scale with
    it exactly as at 1 (a power of two), within the same bounds."""
    x = _inputs()
    scale = 1 / 8.0
    want = R.attention_backward(x["q"], x["k"], x["v"], x["do"], scale, False)
    x[name] = np.ldexp(x[name], power)
    if name in ("q", "k"):
        other = "k" if name == "q" else "q"
        x[other] = np.ldexp(x[other], -power)
    got = _layer(x, scale)
    powers = {"k": {"dq": power, "dk": -power}, "q": {"dk": power, "dq": -power},
              "v": {"o": power, "dq": power, "dk": power},
              "do": {"dq": power, "dk": power, "dv": power}}[name]
    for out in ("o", "lse", "dq", "dk", "dv"):
        back = np.ldexp(got[out].astype(np.float64), -powers.get(out, 0))
        assert T.hybrid_error(back, want[out]) <= 1e-4, out


def test_infinities_stay_in_their_columns(device):
    x = _inputs(seq=100)
    x["v"][0, 7, 3] = np.inf
    got = _layer(x, 1 / 8.0)
    x["v"][0, 7, 3] = 0.0
    want, _, _ = R.attention_forward(x["q"], x["k"], x["v"], 1 / 8.0, False)
    assert np.all(got["o"][0, :, 3] == np.inf)
    keep = np.ones(64, bool)
    keep[3] = False
    assert T.hybrid_error(got["o"][0][:, keep], want[0][:, keep]) <= 2e-5
    assert T.hybrid_error(got["o"][1], want[1]) <= 2e-5


def test_small_probabilities_and_score_gradients(device):
    """P and dS near the bottom of the range from operands that are not: their
    parts keep fp32's bits."""
    x = _inputs()
    scale = 1 / 8.0
    want = R.attention_backward(x["q"], x["k"], x["v"], x["do"], scale, False)
    x["v"], x["do"] = np.ldexp(x["v"], -24), np.ldexp(x["do"], -96)
    got = _layer(x, scale)
    for out, power in {"o": -24, "dq": -120, "dk": -120, "dv": -96}.items():
        assert T.hybrid_error(np.ldexp(got[out].astype(np.float64), -power), want[out]) <= 1e-4, out

    x = _inputs()
    x["q"][:, :, 0] = 8.0
    x["k"][:, :, 0] = 0.0
    x["k"][:, 0] = 0.0
    x["k"][:, 0, 0] = -83.2  # key 0: P of about 2^-125 for every query
    got = _layer(x, scale)
    want = R.attention_backward(x["q"], x["k"], x["v"], x["do"], scale, False)
    small, exact = got["dv"][:, 0].astype(np.float64), want["dv"][:, 0]
    assert np.linalg.norm(exact) < 2.0 ** -105
    assert np.linalg.norm(small - exact) <= 1e-4 * np.linalg.norm(exact)


@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_scores_past_the_scaled_range(device, sign):
    """Scores of 2^100 and a scale that brings them back: the fp32 body."""
    x = _inputs(seq=100)
    want = R.attention_backward(x["q"], x["k"], x["v"], x["do"], sign / 8.0, True)
    x["q"], x["k"] = np.ldexp(x["q"], 50), np.ldexp(x["k"], 50)
    got = _layer(x, sign * 2.0 ** -103, causal=True)
    for out, power in {"o": 0, "lse": 0, "dq": -50, "dk": -50, "dv": 0}.items():
        assert T.hybrid_error(np.ldexp(got[out].astype(np.float64), -power), want[out]) <= 1e-4, out


def test_scores_of_one_product(device):
    """One row, q with one nonzero column and a score scale of one in log2 units: L is
    the rounded product, and O, with P = 1, is V."""
    rng = np.random.default_rng(8)
    heads, dim = 600, 64
    x = _inputs(heads, 1, dim)
    x["q"][...] = 0.0
    x["q"][np.arange(heads), 0, rng.integers(0, dim, heads)] = rng.standard_normal(heads, dtype=np.float32)
    scale = np.float32(np.log(2.0))
    assert scale * np.float32(1.44269504088896340736) == np.float32(1.0)
    got = _layer(x, float(scale))
    exact = np.sum(x["q"][:, 0].astype(np.float64) * x["k"][:, 0], axis=1)
    ulp = np.exp2(np.floor(np.log2(np.abs(exact))) - 23)
    assert np.max(np.abs(got["lse"][:, 0] - exact) / ulp) <= 0.52
    assert np.array_equal(got["o"], x["v"])
