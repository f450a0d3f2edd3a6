"""The weight-row kernel of the 32-element block types on rows that are no multiple of 256
elements (csrc/k_gemmw.hip, k_gemmw_b32): whole stages of 128 in an odd number, a last stage of
one to three blocks, rows that start at 2-byte alignment, a matrix that ends in half a dword (an
odd number of rows of an odd number of blocks), and K splits; against the oracle, and against the
GEMV the calls keep to under graph capture."""
import numpy as np
import pytest

from cllm_inference_amd import synth as S
from test_gpu_parity import check_close, _dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("splits", [0, 2, 3])
@pytest.mark.parametrize("qt", [S.Q8_0, S.Q4_0, S.Q5_0])
def test_rows_of_whole_blocks(gpu, orc, qt, splits):
    for n, k, m in ((300, 896, 100), (1, 32, 17), (129, 416, 33), (255, 2080, 64), (131, 1120, 17),
                    (128, 1056, 31), (257, 160, 65), (64, 4000, 18)):
        if splits > (k + 127) // 128:
            continue
        w = S.make_weight(qt, n, k, n + k)
        x = S.make_activation(m, k, m, outliers=True)
        bias = np.random.default_rng(k).standard_normal(n).astype(np.float32)
        gpu.tune("gemm_splits", splits)
        try:
            print("k32", S.TYPE_NAMES[qt], n, k, m, gpu.matmul_plan(qt, k, n, m), flush=True)
            assert gpu.matmul_route(qt, k, n, m) == "mfma"
            y = gpu.matmul_quant_dev(_dev(x), _dev(w), qt, _dev(bias), k, n).cpu().numpy()
            res = _dev(np.ones((m, n), np.float32))
            if n % 4 == 0:
                gpu.matmul_quant_residual_dev(_dev(x), _dev(w), qt, _dev(bias), k, n, res)
        finally:
            gpu.tune("gemm_splits")
        exact, abs_sum = orc.matmul_f64(x, w, qt, bias, k, n, m)
        yo = orc.matmul(x, w, qt, bias, k, n, m)
        check_close(y, yo, exact, abs_sum, f"{S.TYPE_NAMES[qt]} {n}x{k} m{m} splits={splits}")
        if n % 4 == 0:
            assert np.array_equal(res.cpu().numpy(), 1.0 + y)


def test_rows_of_whole_blocks_under_capture(gpu, orc):
    """A captured call with nothing warmed up but the activation workspace, replayed between eager
    work, has the bits of an eager call whose K is not split (there is no room for partial sums)."""
    import torch
    qt, n, k, m = S.Q8_0, 300, 2080, 48
    w, x = S.make_weight(qt, n, k, 1), S.make_activation(m, k, 2, outliers=True)
    wd, xd = _dev(w), _dev(x)
    eager = gpu.matmul_quant_dev(xd, wd, qt, None, k, n).clone()
    gpu.tune("gemm_splits", 1)
    whole = gpu.matmul_quant_dev(xd, wd, qt, None, k, n).clone()
    gpu.tune("gemm_splits")
    assert not torch.equal(whole, eager)  # split by default
    y = torch.zeros((m, n), device="cuda")
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        # as many activations on a K that is not split: no partial sums are allocated
        assert "splits=1" in gpu.matmul_plan(qt, 896, 1, 120)
        gpu.matmul_quant_dev(_dev(S.make_activation(120, 896, 3)), _dev(S.make_weight(qt, 1, 896, 3)), qt,
                             None, 896, 1)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        gpu.matmul_quant_dev(xd, wd, qt, None, k, n, y=y)
    exact, abs_sum = orc.matmul_f64(x, w, qt, None, k, n, m)
    yo = orc.matmul(x, w, qt, None, k, n, m)
    for rep in range(3):
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        check_close(y.cpu().numpy(), yo, exact, abs_sum, f"replay {rep}")
        assert torch.equal(y, whole), rep
        again = gpu.matmul_quant_dev(xd, wd, qt, None, k, n)
        assert torch.equal(again, eager)


BLOCK_BYTES = {S.Q8_0: 34, S.Q4_0: 18, S.Q5_0: 22}


@pytest.mark.parametrize("splits", [0, 2])
@pytest.mark.parametrize("k", [896, 1120])
@pytest.mark.parametrize("qt", [S.Q8_0, S.Q4_0, S.Q5_0])
def test_rows_of_whole_blocks_infinite_sums(gpu, orc, qt, k, splits):
    """A weight block whose scale is infinite, in an early, a middle and the last stage, makes its
    row's outputs the infinities (or, with an opposite one or a zero block sum, the NaNs) that the
    fp32 sums of the oracle give; the other rows keep the bits they have without it."""
    n, m, nb = 70, 40, k // 32
    w = S.make_weight(qt, n, k, 3)
    x = S.make_activation(m, k, 4)
    bad = w.copy()
    blocks = bad.reshape(n, nb, BLOCK_BYTES[qt])
    for row, blk, bits in ((1, 0, 0x7C00), (7, 0, 0xFC00), (33, 9, 0x7C00), (34, nb - 1, 0x7C00),
                           (50, 5, 0x7E00)):
        blocks[row, blk, :2] = np.frombuffer(np.uint16(bits).tobytes(), np.uint8)
    # two opposite infinities
    for blk, bits in ((2, 0x7C00), (nb - 2, 0xFC00)):
        blocks[60, blk, :2] = np.frombuffer(np.uint16(bits).tobytes(), np.uint8)
    gpu.tune("gemm_splits", splits)
    try:
        assert gpu.matmul_route(qt, k, n, m) == "mfma"
        got = gpu.matmul_quant_dev(_dev(x), _dev(bad), qt, None, k, n).cpu().numpy()
        clean = gpu.matmul_quant_dev(_dev(x), _dev(w), qt, None, k, n).cpu().numpy()
    finally:
        gpu.tune("gemm_splits")
    want = orc.matmul(x, bad, qt, None, k, n, m).reshape(m, n)
    rows = [1, 7, 33, 34, 50, 60]
    assert np.isinf(want[:, [1, 7, 33, 34]]).sum() > 3 * m  # the case holds what it is about
    assert np.array_equal(got[:, rows], want[:, rows], equal_nan=True)
    keep = [r for r in range(n) if r not in rows]
    assert np.array_equal(got[:, keep], clean[:, keep])


@pytest.mark.parametrize("qt", [S.Q8_0, S.Q4_0, S.Q5_0])
def test_rows_of_whole_blocks_infinite_last_activation_scale(gpu, orc, qt):
    """Pre-quantized rows whose last block has an infinite scale, at a K that ends inside a stage:
    the blocks past K add nothing, so the outputs are the GEMV's infinities and NaNs."""
    n, k, m = 40, 1120, 20
    w = _dev(S.make_weight(qt, n, k, 5))
    qs, sc, bs = gpu.quantize_q8_0_dev(_dev(S.make_activation(m, k, 6)))
    sc[3, -1] = float("inf")
    sc[4, 0] = float("inf")
    assert gpu.matmul_route(qt, k, n, m) == "mfma"
    got = gpu.gemv_q8_dev(w, qt, k, n, qs, sc, bs).cpu().numpy()
    # at most 8 rows take the GEMV
    want = np.concatenate([gpu.gemv_q8_dev(w, qt, k, n, qs[t:t + 4].clone(), sc[t:t + 4].clone(),
                                           bs[t:t + 4].clone()).cpu().numpy() for t in range(0, m, 4)])
    assert np.isinf(want[3:5]).any()
    assert np.array_equal(got[3:5], want[3:5], equal_nan=True)
    rest = [t for t in range(m) if t not in (3, 4)]
    np.testing.assert_allclose(got[rest], want[rest], rtol=1e-4, atol=1e-5 * np.abs(want[rest]).max())


def _captured(fn, stream):
    import torch
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=stream):
        fn()
    return g


def test_rows_of_whole_blocks_captured_after_eager_calls(gpu):
    """Pre-quantized and residual calls that the stream ran eagerly before have the same bits in the
    replays of a graph, also after a larger call has outgrown the workspace the graph uses."""
    import torch
    qt, n, k, m = S.Q8_0, 300, 2080, 48
    wd, xd = _dev(S.make_weight(qt, n, k, 1)), _dev(S.make_activation(m, k, 2, outliers=True))
    big_w, big_x = _dev(S.make_weight(qt, 4096, k, 3)), _dev(S.make_activation(2000, k, 4))
    y, res, s = torch.zeros((m, n), device="cuda"), torch.zeros((m, n), device="cuda"), torch.cuda.Stream()
    qs, sc, bs = gpu.quantize_q8_0_dev(xd)
    assert gpu.matmul_route(qt, k, n, m) == "mfma"
    torch.cuda.synchronize()

    def calls():
        gpu.gemv_q8_dev(wd, qt, k, n, qs, sc, bs, y=y)
        gpu.matmul_quant_residual_dev(xd, wd, qt, None, k, n, res)
    with torch.cuda.stream(s):
        calls()
        eager = (y.clone(), res.clone())
    g = _captured(calls, s)
    for rep in range(4):
        y.zero_(), res.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, eager[0]) and torch.equal(res, eager[1]), rep
        with torch.cuda.stream(s):  # eager work between the replays; the second one grows the workspace
            mm = m if rep == 0 else 2000
            out = torch.zeros((mm, 4096), device="cuda")
            gpu.matmul_quant_residual_dev(big_x[:mm].contiguous(), big_w, qt, None, k, 4096, out)
        torch.cuda.synchronize()


def test_rows_of_whole_blocks_captured_without_room(gpu, orc):
    """The same calls captured on a stream whose workspace has no room for them (no pre-quantized call
    and no residual buffer before) take the GEMV, which allocates nothing."""
    import torch
    qt, n, k, m = S.Q8_0, 300, 2080, 48
    w, x = S.make_weight(qt, n, k, 1), S.make_activation(m, k, 2, outliers=True)
    wd, xd, s = _dev(w), _dev(x), torch.cuda.Stream()
    y, res, fresh = torch.zeros((m, n), device="cuda"), torch.zeros((m, n), device="cuda"), torch.cuda.Stream()
    qs, sc, bs = gpu.quantize_q8_0_dev(xd)
    with torch.cuda.stream(s):
        gpu.matmul_quant_dev(xd, wd, qt, None, k, n)  # activations and partial sums, no residual buffer
    g1 = _captured(lambda: gpu.gemv_q8_dev(wd, qt, k, n, qs, sc, bs, y=y), fresh)
    g2 = _captured(lambda: gpu.matmul_quant_residual_dev(xd, wd, qt, None, k, n, res), s)
    want = np.concatenate([gpu.gemv_q8_dev(wd, qt, k, n, qs[t:t + 8].clone(), sc[t:t + 8].clone(),
                                           bs[t:t + 8].clone()).cpu().numpy() for t in range(0, m, 8)])
    exact, abs_sum = orc.matmul_f64(x, w, qt, None, k, n, m)
    yo = orc.matmul(x, w, qt, None, k, n, m)
    check_close(want, yo, exact, abs_sum, "GEMV")
    for rep in range(3):
        y.zero_(), res.zero_()
        g1.replay(), g2.replay()
        torch.cuda.synchronize()
        assert np.array_equal(y.cpu().numpy(), want) and np.array_equal(res.cpu().numpy(), want), rep
        gpu.matmul_quant_dev(xd, wd, qt, None, k, n)
