"""Each kernel for int8 rows on re-tiled filters at sizes that are asked for first
(lrtfc_fc_int8_packed_kernel), so that a change of the dispatch rules cannot leave one of them, or
one of its forms, without a test. Bit-exact against the CPU oracle."""
import numpy as np
import pytest

import oracle
from litert_amd import capi
from litert_amd import workloads as wl
from tests.test_gpu_parity import _bits_equal, _cuda, _run_int8, fc  # noqa: F401

pytestmark = pytest.mark.gpu

GEMV, TWO, ROWS, SPLIT, T64, T128 = (
    capi.INT8_KERNEL_GEMV, capi.INT8_KERNEL_GEMV_TWO_TILES, capi.INT8_KERNEL_ROWS,
    capi.INT8_KERNEL_SPLIT, capi.INT8_KERNEL_TILES_64X128, capi.INT8_KERNEL_TILES_128X256)

SHAPES = [
    # one row tile: shares of up to 8, 16 and 32 tiles, rows of one to 16 pieces a thread, whole
    # rows and rows that end inside a piece; the refilled ring, rows in registers and not
    (GEMV, 9, 512, 40), (GEMV, 16, 1024, 40), (GEMV, 15, 1021, 40), (GEMV, 9, 2048, 8200),
    (GEMV, 16, 2047, 8200), (GEMV, 16, 4096, 8200), (GEMV, 9, 4093, 8200), (GEMV, 2, 8190, 70),
    (GEMV, 8, 8192, 70), (GEMV, 7, 8177, 70), (GEMV, 4, 16384, 9), (GEMV, 3, 16381, 9),
    (GEMV, 4, 20016, 9), (GEMV, 4, 20003, 9), (GEMV, 9, 8192, 8200), (GEMV, 8, 8203, 8200),
    # two row tiles: the same shares
    (TWO, 17, 512, 16400), (TWO, 32, 1022, 16400), (TWO, 32, 2048, 16400), (TWO, 18, 2047, 16400),
    (TWO, 17, 4096, 8193), (TWO, 32, 4093, 8200),
    # the rows kernel with four row tiles and with eight; odd and even numbers of depth chunks
    (ROWS, 33, 1024, 16400), (ROWS, 64, 1037, 16400), (ROWS, 48, 1300, 16400), (ROWS, 33, 2047, 16400),
    (ROWS, 65, 1024, 10241), (ROWS, 128, 1037, 10241), (ROWS, 97, 1535, 10250),
    # small tiles: at the row counts and depths that still go there up to 16 rows, and beyond
    (SPLIT, 16, 4100, 255), (SPLIT, 12, 8208, 33), (SPLIT, 7, 20000, 40), (SPLIT, 9, 1040, 6200),
    (SPLIT, 17, 16, 5), (SPLIT, 24, 129, 33), (SPLIT, 31, 2112, 67), (SPLIT, 64, 1024, 10300),
    (T64, 130, 1024, 10240), (T64, 200, 1037, 8200), (T128, 1100, 131, 4099),
]


def _check_kernel(kernel, B, K, N):
    assert capi.load().lrtfc_fc_int8_packed_kernel(B, K, N) == kernel


@pytest.mark.parametrize("kernel,B,K,N", SHAPES)
def test_int8_on_its_kernel(fc, kernel, B, K, N):  # noqa: F811
    _check_kernel(kernel, B, K, N)
    y, want = _run_int8(fc, wl.int8_fc(B, K, N, in_zp=(-3 if K % 2 else 0), seed=B + K + N),
                        "relu6" if N % 2 else "none", bias=B % 2 == 0)
    assert np.array_equal(y, want)


@pytest.mark.parametrize("kernel,B,K,N", SHAPES)
def test_hybrid_on_its_kernel(fc, kernel, B, K, N):  # noqa: F811
    """Through the row quantizer, whose rows are padded: both quantizations, bias elements of -0.0f,
    and a whole-zero input, which keeps their sign."""
    _check_kernel(kernel, B, (K + 15) // 16 * 16, N)
    c = wl.hybrid_fc(B, K, N, seed=B + K + N)
    bias = np.random.default_rng(K).standard_normal(N).astype(np.float32)
    bias[::5] = -0.0
    for asym in ((True, False) if B * K * N < 3e8 else (bool(B % 2),)):
        op = fc.FullyConnectedHybrid(c["w"], c["pcs"], bias=bias, asymmetric_quantize_inputs=asym)
        want = oracle.fc_hybrid(c["x"], c["w"], c["pcs"], bias=bias, asymmetric=asym)
        assert _bits_equal(op.call_split(_cuda(c["x"])).cpu().numpy(), want)
        zeros = np.zeros_like(c["x"])
        want = oracle.fc_hybrid(zeros, c["w"], c["pcs"], bias=bias, asymmetric=asym)
        assert _bits_equal(op.call_split(_cuda(zeros)).cpu().numpy(), want)


@pytest.mark.parametrize("kernel,B,K,N", [s for s in SHAPES if s[2] % 16])
def test_hybrid_rows_that_arrive_quantized(fc, kernel, B, K, N):  # noqa: F811
    """The caller's own rows, not padded: they end inside a 16-byte piece."""
    import torch
    _check_kernel(kernel, B, K, N)
    c = wl.hybrid_fc(B, K, N, seed=B + K + N)
    op = fc.FullyConnectedHybrid(c["w"], c["pcs"])
    q, sf, zp = oracle.batch_quantize_floats(c["x"], True)
    dq, dsf, dzp = _cuda(q), _cuda(sf), _cuda(zp.astype(np.int32))
    out = torch.empty((B, N), device="cuda")
    ptr = lambda t: t.data_ptr()  # noqa: E731
    capi.check(capi.load().lrtfc_fc_hybrid_int8_packed(
        ptr(dq), ptr(dsf), ptr(dzp), ptr(op.packed_filter), ptr(op.pcs), 1.0, ptr(op.row_sums), None,
        ptr(out), B, K, N, 0, torch.cuda.current_stream().cuda_stream))
    assert _bits_equal(out.cpu().numpy(), oracle.fc_hybrid(c["x"], c["w"], c["pcs"]))
