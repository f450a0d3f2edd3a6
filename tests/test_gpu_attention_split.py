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


@pytest.mark.parametrize("hd,n_head,n_kv", [(64, 8, 2), (128, 8, 2), (64, 4, 4), (128, 14, 2), (128, 5, 5)])
@pytest.mark.parametrize("rows,pos0", [(96, 20), (130, 0), (40, 300)])
def test_split_attention_non_finite_columns(gpu, hd, n_head, n_kv, rows, pos0):
    """Infinities and NaN in queries, keys and values: each column has the infinities and NaNs of the
    same in 64 bits, and a column that meets none of them keeps its bits, also beside columns of its
    workgroup that do. (Columns of a row block that holds the first row to see such a value meet it
    with a probability of zero and are computed again.)"""
    rng = np.random.default_rng(hd + n_head + rows)
    L, rep = pos0 + rows, n_head // n_kv
    q = rng.standard_normal((rows, n_head, hd)).astype(np.float32)
    kc = rng.standard_normal((L, n_kv, hd)).astype(np.float32)
    vc = rng.standard_normal((L, n_kv, hd)).astype(np.float32)
    qb, kb, vb = q.copy(), kc.copy(), vc.copy()
    touched = np.zeros((rows, n_head), bool)
    for t, h, val in ((3, 0, np.nan), (rows - 1, n_head - 1, np.inf), (rows // 2, 1, 3.4e38)):
        qb[t, h, 5] = val
        touched[t, h] = True
    # scores of minus infinity (no weight) or infinity (NaN) by the query's sign; a NaN key; values
    for arr, pos, g, dim, val in ((kb, L - 30, 0, 1, np.inf), (kb, L - 9, 0, 2, np.nan),
                                  (vb, L - 25, n_kv - 1, 7, np.inf), (vb, L - 21, n_kv - 1, 9, -np.inf),
                                  (vb, L - 13, n_kv - 1, 11, np.nan), (vb, L - 12, n_kv - 1, 13, 3.4e38)):
        arr[pos, g, dim] = val
        first = max(pos - pos0, 0) // (32 // rep) * (32 // rep)
        touched[first:, g * rep:(g + 1) * rep] = True
    args = (pos0, n_head, n_kv, hd)
    gpu.tune("attention_kernel", 2)
    try:
        got = gpu.attention_dev(_dev(qb.reshape(rows, -1)), _dev(kb.reshape(L, -1)), _dev(vb.reshape(L, -1)),
                                *args).cpu().numpy().reshape(rows, n_head, hd)
        clean = gpu.attention_dev(_dev(q.reshape(rows, -1)), _dev(kc.reshape(L, -1)), _dev(vc.reshape(L, -1)),
                                  *args).cpu().numpy().reshape(rows, n_head, hd)
    finally:
        gpu.tune("attention_kernel")
    assert touched.any() and not touched.all()
    assert np.array_equal(got[~touched], clean[~touched])
    with np.errstate(all="ignore"):
        want = _attn_ref(qb.reshape(rows, -1), kb.reshape(L, -1), vb.reshape(L, -1), *args).reshape(got.shape)
    # (scores past 3.4e38 overflow in 32 bits: that column is NaN or one position's values)
    want[rows // 2, 1] = got[rows // 2, 1]
    assert np.array_equal(np.isnan(got), np.isnan(want))
    inf = np.isinf(want)
    assert inf.any() and np.array_equal(got[inf], want[inf])
    fin = np.isfinite(want)
    np.testing.assert_allclose(got[fin], want[fin], rtol=2e-5, atol=2e-5)


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("q_exp,k_exp,v_exp", [(-116, 114, 0), (114, -116, 0), (0, 0, -116), (0, 0, 110),
                                               (-60, 60, -95)])
def test_split_attention_small_and_large_values(gpu, hd, q_exp, k_exp, v_exp):
    """Queries, keys and values far from 1, whose lower bf16 parts the matrix cores would take for zero:
    as near to the same in 64 bits as values around 1 (2e-6 of the largest output; without a measure
    against it 1e-5 and up). (Values of 2^-6 to 2 before the scaling: none is below the smallest
    normal fp32.)"""
    rng = np.random.default_rng(hd + abs(v_exp))
    n_head, n_kv, rows, pos0 = 8, 2, 70, 50
    def draw(r, c):
        return (rng.uniform(2.0 ** -6, 2, (r, c)) * rng.choice([-1, 1], (r, c))).astype(np.float32)
    q, k, v = draw(rows, n_head * hd), draw(pos0 + rows, n_kv * hd), draw(pos0 + rows, n_kv * hd)
    two = np.float32(2.0)
    gpu.tune("attention_kernel", 2)
    try:
        got = gpu.attention_dev(_dev(q * two ** q_exp), _dev(k * two ** k_exp), _dev(v * two ** v_exp), pos0,
                                n_head, n_kv, hd).cpu().numpy().astype(np.float64) * 2.0 ** -v_exp
    finally:
        gpu.tune("attention_kernel")
    want = _attn_ref(q * two ** (q_exp + k_exp), k, v, pos0, n_head, n_kv, hd)
    assert (np.abs(got - want) <= 2e-6 * np.abs(want).max()).all(), np.abs(got - want).max()


def test_split_attention_zero_values(gpu):
    """Value dims that are all zero (padding) stay zero."""
    rng = np.random.default_rng(1)
    q, k, v = (rng.standard_normal((r, c * 128)).astype(np.float32) for r, c in ((64, 8), (200, 2), (200, 2)))
    v.reshape(200, 2, 128)[:, :, 80:] = 0.0
    gpu.tune("attention_kernel", 2)
    try:
        got = gpu.attention_dev(_dev(q), _dev(k), _dev(v), 136, 8, 2, 128).cpu().numpy().reshape(64, 8, 128)
    finally:
        gpu.tune("attention_kernel")
    assert not got[:, :, 80:].any() and (got[:, :, :80] != 0).all()


def test_attention_caches_past_4_gib(gpu):
    """The fp32 MFMA form at head_dim 64 and 128, which caches of 4 GiB and more take (32-bit offsets
    in the other), at every number of heads per KV head it lays out differently: the last rows of a
    long cache against the sequence-split kernel on the same rows and against the same in 64 bits for
    a few heads. The softmax of 130000 positions: sums of fp32 rounding 2^-24 sqrt(130000) of the
    mean value, 3e-5 of the largest output."""
    import torch
    if torch.cuda.get_device_properties(0).total_memory < 48 << 30:
        pytest.skip("needs 48 GiB of GPU memory")
    g = torch.Generator(device="cuda").manual_seed(3)
    for hd, n_kv in ((128, 64), (64, 128)):
        L = (1 << 32) // (n_kv * hd * 4) + 117  # 4 GiB and 117 rows
        k = torch.randn((L, n_kv * hd), device="cuda", generator=g)
        v = torch.randn((L, n_kv * hd), device="cuda", generator=g)
        for rep, rows in ((1, 1), (1, 40), (3, 33), (4, 17), (8, 70)):
            n_head, pos0 = n_kv * rep, L - rows
            q = torch.randn((rows, n_head * hd), device="cuda", generator=g)
            print("attention past 4 GiB", hd, n_kv, rep, rows, flush=True)
            gpu.tune("attention_kernel", 2)
            try:
                assert gpu.attention_plan(rows, pos0, n_head, n_kv, hd).startswith(f"k_attention_mfma_f32<{hd}")
                got = gpu.attention_dev(q, k, v, pos0, n_head, n_kv, hd)
                gpu.tune("attention_kernel", 1)
                other = gpu.attention_dev(q, k, v, pos0, n_head, n_kv, hd)
            finally:
                gpu.tune("attention_kernel")
            assert (got - other).abs().max() <= 3e-5 * other.abs().max(), (hd, rep, rows)
            got = got.view(rows, n_head, hd)
            for h in (0, n_head // 2, n_head - 1):
                kv = slice(h // rep * hd, (h // rep + 1) * hd)
                s = q.view(rows, n_head, hd)[:, h].double() @ k[:, kv].double().T.contiguous() / hd ** 0.5
                seen = torch.arange(L, device="cuda")[None] <= pos0 + torch.arange(rows, device="cuda")[:, None]
                want = torch.softmax(s.masked_fill(~seen, float("-inf")), -1) @ v[:, kv].double()
                assert (got[:, h] - want).abs().max() <= 3e-5 * want.abs().max(), (hd, rep, rows, h)
        del k, v


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


def test_captured_attention_outlives_its_workspace(gpu):
    """A batch of one head per KV head on the sequence-split kernel, captured after an eager call, keeps
    its bits in replays after a larger call on the stream has outgrown the split partials' workspace."""
    import torch
    hd, heads, rows, pos0 = 128, 8, 64, 1024
    assert gpu.attention_plan(rows, pos0, heads, heads, hd).startswith("k_attention<")
    g = torch.Generator(device="cuda").manual_seed(2)
    q, k, v = (torch.randn((r, heads * hd), device="cuda", generator=g) for r in (rows, pos0 + rows, pos0 + rows))
    big = torch.randn((2048, 32 * hd), device="cuda", generator=g)
    out, s = torch.zeros_like(q), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        eager = gpu.attention_dev(q, k, v, pos0, heads, heads, hd).clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        gpu.attention_dev(q, k, v, pos0, heads, heads, hd, out=out)
    for rep in range(4):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager), rep
        with torch.cuda.stream(s):  # the workspace is sized by rows and heads: 2048 rows outgrow it
            n = 64 if rep == 0 else 2048
            gpu.attention_dev(big[:n].contiguous(), big[:n, :8 * hd].contiguous(), big[:n, :8 * hd].contiguous(),
                              0, 32, 8, hd)
        torch.cuda.synchronize()
