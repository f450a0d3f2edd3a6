"""The split-operand MFMA kernel of the float-dot types (csrc/k_gemm_f.hip) against the 64-bit
sums, on every tile shape: weight rows and tokens at the edges of tiles, K of an odd number of
32-element units, of less than a 256-element chunk and of a chunk more than the waves share
evenly. Bars as for the GEMV of these types (test_gpu_fdot.py)."""
import numpy as np
import pytest

from cllm_inference_amd import synth as S
from test_gpu_parity import check_close, _dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [1, 2, 3])
@pytest.mark.parametrize("qt", list(S.FLOAT_DOT_TYPES))
def test_split_operand_gemm_edges(gpu, orc, qt, shape):
    step = max(S.BLOCK[qt], 32)
    for n, units, m in ((1, 1, 8), (31, 3, 33), (33, 9, 2), (129, 5, 65), (70, 27, 31), (128, 8, 64)):
        k = step * units
        w = S.make_weight(qt, n, k, 7 * n + k)
        x = S.make_activation(m, k, m + k, outliers=True)
        bias = np.random.default_rng(n).standard_normal(n).astype(np.float32)
        print("gemm_f", S.TYPE_NAMES[qt], "shape", shape, n, k, m, flush=True)
        gpu.tune("gemm_f", shape)
        try:
            y = gpu.matmul_quant_dev(_dev(x), _dev(w), qt, _dev(bias), k, n).cpu().numpy()
        finally:
            gpu.tune("gemm_f")
        exact, abs_sum = orc.matmul_f64(x, w, qt, bias, k, n, m)
        yo = orc.matmul(x, w, qt, bias, k, n, m).reshape(m, n)
        check_close(y, yo, exact, abs_sum, f"{S.TYPE_NAMES[qt]} shape {shape} {n}x{k} m{m}")


@pytest.mark.parametrize("qt", list(S.FLOAT_DOT_TYPES))
def test_split_operand_gemm_non_finite(gpu, orc, qt):
    """Activations with infinities, NaN and values past the largest bf16 give the reference's
    infinities and NaNs, and the rows beside them the values of a batch without them."""
    k, n, m = 512, 40, 12
    w = S.make_weight(qt, n, k, 3)
    x = S.make_activation(m, k, 4)
    clean = x.copy()
    x[1, 5], x[4, 300], x[7, 17], x[9, 2] = np.inf, -np.inf, np.nan, 3.4e38
    out = {}
    for knob in (1, 2, 3):
        gpu.tune("gemm_f", knob)
        try:
            out[knob] = gpu.matmul_quant_dev(_dev(x), _dev(w), qt, None, k, n).cpu().numpy()
            if knob == 2:
                beside = gpu.matmul_quant_dev(_dev(clean), _dev(w), qt, None, k, n).cpu().numpy()
        finally:
            gpu.tune("gemm_f")
    ref = orc.matmul(x, w, qt, None, k, n, m).reshape(m, n)
    for knob in (1, 2, 3):
        y = out[knob]
        for t in (1, 4, 7):
            # a zero weight makes inf * 0 = NaN; the others keep the sign
            assert np.array_equal(np.isnan(y[t]), np.isnan(ref[t])), (knob, t)
            inf = np.isinf(ref[t])
            assert np.array_equal(y[t][inf], ref[t][inf]), (knob, t)
        fin = np.isfinite(ref[9])
        assert np.array_equal(np.isfinite(y[9]), fin), knob
        np.testing.assert_allclose(y[9][fin], ref[9][fin], rtol=1e-5)
    rows = [t for t in range(m) if t not in (1, 4, 7, 9)]
    assert np.array_equal(out[2][rows], beside[rows])


@pytest.mark.parametrize("k_units", [1, 9, 16])
@pytest.mark.parametrize("qt", list(S.FLOAT_DOT_TYPES))
def test_split_operand_gemm_infinite_weights(gpu, orc, qt, k_units):
    """Weights that decode to infinity or NaN, in tiles with rows and tokens past the matrix: the
    reference's infinities and NaNs in their outputs, and no other output changed."""
    n, m, k = 40, 37, max(S.BLOCK[qt], 32) * k_units
    w = S.make_weight(qt, n, k, 3)
    x = S.make_activation(m, k, 4)
    bad = w.copy()
    rows = bad.reshape(n, -1)
    at = {S.Q2_K: 80, S.Q3_K: 108}.get(qt, 0)  # the scale of the row's first block
    for row, half, single in ((5, 0x7C00, np.inf), (31, 0xFC00, -np.inf), (39, 0x7E00, np.nan)):
        raw = np.float32(single).tobytes() if qt == S.F32 else np.uint16(half).tobytes()
        rows[row, at:at + len(raw)] = np.frombuffer(raw, np.uint8)
    ref = orc.matmul(x, bad, qt, None, k, n, m).reshape(m, n)
    hit = [5, 31, 39]
    assert not np.isfinite(ref[:, hit]).any()
    for knob in (1, 2, 3):
        gpu.tune("gemm_f", knob)
        try:
            y = gpu.matmul_quant_dev(_dev(x), _dev(bad), qt, None, k, n).cpu().numpy()
            clean = gpu.matmul_quant_dev(_dev(x), _dev(w), qt, None, k, n).cpu().numpy()
        finally:
            gpu.tune("gemm_f")
        assert np.array_equal(y[:, hit], ref[:, hit], equal_nan=True), knob
        keep = [r for r in range(n) if r not in hit]
        assert np.array_equal(y[:, keep], clean[:, keep]), knob


@pytest.mark.parametrize("qt,w_exp,x_exp", [(S.F32, -120, 115), (S.F32, 112, -118), (S.F32, -60, -55),
                                            (S.F16, 0, -118), (S.Q4_1, 0, -118), (S.Q8_1, 0, -118),
                                            (S.Q2_K, 0, -115), (S.Q3_K, 0, -115), (S.Q5_1, 0, 90)])
def test_split_operand_gemm_small_and_large_values(gpu, qt, w_exp, x_exp):
    """Weights and activations far from 1, whose lower bf16 parts the matrix cores would take for zero:
    as near to the 64-bit sums as batches around 1. (Values of 2^-6 to 1 before the scaling: none is
    below the smallest normal fp32. 512 terms of random sign: sums of fp32 rounding, 3e-7 of the
    result's norm at most; without the scaling 1e-5 and up.)"""
    import torch
    n, m, k = 96, 40, 512
    rng = np.random.default_rng(qt)
    x = (rng.uniform(2.0 ** -6, 1, (m, k)) * rng.choice([-1, 1], (m, k))).astype(np.float32)
    if qt == S.F32:
        w = (rng.uniform(2.0 ** -6, 1, (n, k)) * rng.choice([-1, 1], (n, k))).astype(np.float32)
        full = w.astype(np.float64)
        w = (w * np.float32(2.0) ** w_exp).view(np.uint8).reshape(-1)
    else:
        w = S.make_weight(qt, n, k, 3)
        full = gpu.dequantize_rows_dev(_dev(w), qt, k, torch.arange(n, device="cuda", dtype=torch.int32))
        full = full.double().cpu().numpy().reshape(n, k)
    want = x.astype(np.float64) @ full.T
    xs = _dev(x * np.float32(2.0) ** x_exp)
    for knob in (1, 2, 3):
        gpu.tune("gemm_f", knob)
        try:
            y = gpu.matmul_quant_dev(xs, _dev(w), qt, None, k, n).double().cpu().numpy()
        finally:
            gpu.tune("gemm_f")
        err = y * 2.0 ** -(w_exp + x_exp) - want
        assert np.linalg.norm(err) <= 3e-7 * np.linalg.norm(want), (knob, np.linalg.norm(err) / np.linalg.norm(want))
