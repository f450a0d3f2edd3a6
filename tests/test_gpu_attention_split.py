"""The prefill attention's split operands (csrc/k_attention.hip, k_attention_mfma at head_dim 64 and
128): steps of 32 positions at the edges (1 to 65 positions, a wave that straddles two row blocks,
waves without work), values over a wide range, and inputs that are not finite; and the decode
kernel at its edges."""
import numpy as np
import pytest

from test_gpu_attention import _attn_ref
from test_gpu_parity import _dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd,n_head,n_kv", [(128, 8, 2), (64, 7, 1), (128, 5, 5)])
@pytest.mark.parametrize("rows,pos0", [(1, 0), (31, 0), (33, 0), (5, 27), (9, 56), (40, 479)])
def test_split_attention_edges(gpu, hd, n_head, n_kv, rows, pos0):
    rng = np.random.default_rng(hd + n_head + rows + pos0)
    L = pos0 + rows
    q = (rng.standard_normal((rows, n_head * hd)) * 2.0).astype(np.float32)
    kc = (rng.standard_normal((L, n_kv * hd)) * np.exp(rng.uniform(-6, 1, (L, 1)))).astype(np.float32)
    vc = (rng.standard_normal((L, n_kv * hd)) * np.exp(rng.uniform(-6, 6, (L, 1)))).astype(np.float32)
    gpu.tune("attention_kernel", 2)
    try:
        got = gpu.attention_dev(_dev(q), _dev(kc), _dev(vc), pos0, n_head, n_kv, hd).cpu().numpy()
    finally:
        gpu.tune("attention_kernel")
    want = _attn_ref(q, kc, vc, pos0, n_head, n_kv, hd)
    err = np.abs(got - want).reshape(rows, n_head, hd).max(axis=2)
    scale = np.abs(want).reshape(rows, n_head, hd).max(axis=2)
    # fp32 scores of up to 200 (rounded by 2^-24 of that) in the exponent, then fp32 sums
    assert (err <= 2e-5 * np.maximum(scale, 1e-3)).all(), (err / scale).max()


def test_split_attention_non_finite(gpu):
    """An infinite value row makes its column's outputs infinite from the first row that sees it
    on, with the sign; rows before it, and other KV heads, are as without it."""
    rng = np.random.default_rng(3)
    hd, n_head, n_kv, rows, pos0 = 128, 8, 2, 96, 20
    L = pos0 + rows
    q = rng.standard_normal((rows, n_head * hd)).astype(np.float32)
    kc = rng.standard_normal((L, n_kv * hd)).astype(np.float32)
    vc = rng.standard_normal((L, n_kv * hd)).astype(np.float32)
    bad = vc.copy()
    bad[60, 7], bad[60, 9], bad[60, 11] = np.inf, -np.inf, 3.4e38
    gpu.tune("attention_kernel", 2)
    try:
        want = gpu.attention_dev(_dev(q), _dev(kc), _dev(vc), pos0, n_head, n_kv, hd).cpu().numpy()
        got = gpu.attention_dev(_dev(q), _dev(kc), _dev(bad), pos0, n_head, n_kv, hd).cpu().numpy()
    finally:
        gpu.tune("attention_kernel")
    got, want = (a.reshape(rows, n_head, hd) for a in (got, want))
    assert (got[40:, :4, 7] == np.inf).all() and (got[40:, :4, 9] == -np.inf).all()
    assert np.isfinite(got[40:, :4, 11]).all() and (got[40:, :4, 11] > 1e30).all()
    keep = [d for d in range(hd) if d not in (7, 9, 11)]
    np.testing.assert_allclose(got[:, :, keep], want[:, :, keep], rtol=2e-5, atol=1e-6)
    assert np.array_equal(got[:, 4:], want[:, 4:])


@pytest.mark.parametrize("hd,n_head,n_kv", [(128, 4, 2), (256, 4, 2), (64, 2, 1), (256, 8, 1), (256, 4, 1),
                                            (64, 3, 3), (128, 6, 1)])
def test_decode_attention_edges(gpu, hd, n_head, n_kv):
    """The sequence-split kernel at every number of scores per lane row (one to eight heads per KV
    head, every head_dim): positions at the edges of a wave's step, of a workgroup's four steps and
    of a split, one row and three, against the same in 64 bits."""
    rng = np.random.default_rng(hd + 10 * n_head + n_kv)
    gpu.tune("attention_kernel", 1)
    try:
        for pos0 in (0, 1, 3, 7, 15, 16, 31, 62, 63, 64, 129, 700):
            for rows in (1, 3):
                L = pos0 + rows
                q = rng.standard_normal((rows, n_head * hd)).astype(np.float32)
                kc = rng.standard_normal((L, n_kv * hd)).astype(np.float32)
                vc = rng.standard_normal((L, n_kv * hd)).astype(np.float32)
                got = gpu.attention_dev(_dev(q), _dev(kc), _dev(vc), pos0, n_head, n_kv, hd).cpu().numpy()
                want = _attn_ref(q, kc, vc, pos0, n_head, n_kv, hd)
                err = np.abs(got - want).reshape(rows, n_head, hd).max(axis=2)
                scale = np.abs(want).reshape(rows, n_head, hd).max(axis=2)
                # scores of up to 5, rounded by 2^-24 of that (3e-7) in the exponent and as much in
                # their partial sums, then expf and the output sums (1e-7 each); twice that and more
                assert (err <= 2e-6 * np.maximum(scale, 1e-3)).all(), (pos0, rows, err.max())
    finally:
        gpu.tune("attention_kernel")
