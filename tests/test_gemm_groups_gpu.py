"""16-bit GEMMs whose K loop is split over wave groups inside the workgroup:
every layout, whole and ragged tiles, step counts that leave groups idle in the
last round, and the SAE encoder, against fp64 (operand padding poisoned)."""

import numpy as np
import pytest

from oracle import reference as R
from oracle import tolerance as T
from test_fast_paths_gpu import _gemm, _gemm_nt, _gemm_tn
from triton_metal import _core, ops
from triton_metal.buffer import round_to

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("element", ["bf16", "f16"])
@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
@pytest.mark.parametrize("m,n,k,pad,kernel", [
    (512, 256, 192, 8, "fast{}_t64_k4"),        # 3 steps over 4 groups
    (1280, 1280, 320, 8, "fast{}_t64_k2"),      # 400 tiles, 5 steps over 2
    (2048, 2048, 192, 8, "fast{}_t128_k2"),     # 3 steps over 2
    (576, 640, 4096, 8, "fast{}_t64_k4_ks"),    # groups and ranges
    (520, 776, 200, 8, "ragged{}_t64"),         # 4 groups, the last step ragged
    (511, 513, 321, 7, "ragged{}_t64"),         # 6 steps: the last in the second round
    (1201, 1207, 265, 7, "ragged{}_t64"),       # 2 groups
    (40, 72, 130, 6, "ragged{}_t64"),           # few tiles, few steps
    (500, 1000, 4040, 8, "ragged{}_t64_k4_ks"),
    (257, 511, 321, 1, "generic"),              # unaligned rows
    (1217, 1217, 321, 1, "generic"),
    (511, 1023, 4033, 1, "unaligned{}_t64_k4_ks"),
])
def test_k_groups(device, element, layout, m, n, k, pad, kernel):
    # `pad` past each stored row, to a multiple of 8 except for the unaligned
    up = (lambda x: x + 1 + (x % 2)) if pad == 1 else (lambda x: -(-(x + 1) // 8) * 8)
    if layout == "nn":
        c, want, got = _gemm(m, n, k, element, up(k), up(n), up(n), poison=True, extra_rows=3)
    elif layout == "nt":
        c, want, got = _gemm_nt(m, n, k, element, up(k), up(k), up(n))
    else:
        c, want, got = _gemm_tn(m, n, k, element, up(m), up(n), up(n))
    kernel = kernel.format("" if layout == "nn" else "_" + layout)
    assert got.split(" + ")[0] == f"tm_gemm_{kernel}_{element}"
    assert np.all(np.isfinite(c[:m, :n]))
    assert T.hybrid_error(c[:m, :n], want) <= 2e-2
    assert np.all(c[:m, n:] == -7.0) and np.all(c[m:] == -7.0)


@pytest.mark.parametrize("rows,model,features,kernel", [
    (128, 320, 256, "fast_t64"), (1280, 256, 1280, "fast_t64"), (2048, 192, 2048, "fast_t128"),
    (100, 328, 264, "ragged_t64"), (1920, 256, 2112, "fast_t64_g1"), (2048, 64, 4096, "fast_t128_g1"), (2320, 64, 1032, "ragged_t64_g1"),
    (33, 321, 129, "generic"), (1217, 321, 1217, "generic"),
])
def test_sae_k_groups(device, rows, model, features, kernel):
    rng = np.random.default_rng(5)
    x = round_to(rng.standard_normal((rows, model), dtype=np.float32), "bf16")
    w = round_to(rng.standard_normal((model, features), dtype=np.float32) / np.sqrt(model), "bf16")
    b = round_to(rng.standard_normal(features, dtype=np.float32), "bf16")
    enc = ops.SAEEncoder("bf16")
    got = enc.numpy(x, w, b)
    variant = _core.kernel_variant(enc.kernel)
    assert T.hybrid_error(got, R.sae_encode(x, w, b)) <= 2e-2, variant
    assert variant == f"tm_sae_{kernel}_bf16"


@pytest.mark.parametrize("element", ["bf16", "f16"])
@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
@pytest.mark.parametrize("m,n,k", [(16, 20000, 1024), (63, 16460, 901)])
def test_k_ranges_of_more_tiles_than_compute_units(device, element, layout, m, n, k):
    up = lambda x: -(-(x + 1) // 8) * 8
    if layout == "nn":
        c, want, got = _gemm(m, n, k, element, up(k), up(n), up(n), poison=True, extra_rows=3)
    elif layout == "nt":
        c, want, got = _gemm_nt(m, n, k, element, up(k), up(k), up(n))
    else:
        c, want, got = _gemm_tn(m, n, k, element, up(m), up(n), up(n))
    suffix = "" if layout == "nn" else "_" + layout
    assert got.split(" + ")[0] == f"tm_gemm_ragged{suffix}_t64_ks_{element}"
    assert np.all(np.isfinite(c[:m, :n]))
    assert T.hybrid_error(c[:m, :n], want) <= 2e-2
    assert np.all(c[:m, n:] == -7.0) and np.all(c[m:] == -7.0)
