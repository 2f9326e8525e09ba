"""Depths and channel counts off every vector size, on each kernel that reads rows in 16-byte
pieces: the last piece of a row is read early and shifted into place, and nothing behind a row's
last value may reach a result. Bit-exact against the CPU oracle, as everywhere on these paths."""
import numpy as np
import pytest

import oracle
from litert_amd import capi
from litert_amd import workloads as wl
from tests.test_gpu_parity import _bits_equal, _cuda, _run_int8, fc  # noqa: F401

pytestmark = pytest.mark.gpu

# GEMV (1, 3 and 5 rows), small tiles (16 to 77, 150 and 257 rows), the rows kernel (128 x 10241), large
# GEMM tiles (1100 x 4099). test_gpu_int8_kernels.py has such depths for every kernel, by name.
SHAPES = [(1, 17, 19), (1, 2999, 530), (5, 2049, 67), (16, 1030, 33), (3, 20001, 9), (17, 2047, 301),
          (32, 4093, 515), (77, 1999, 261), (150, 21, 130), (257, 1283, 515), (40, 1027, 10243),
          (128, 1037, 10241), (1100, 131, 4099)]


@pytest.mark.parametrize("B,K,N", SHAPES)
@pytest.mark.parametrize("activation", ["none", "relu6"])
def test_int8_ragged_depth_bit_exact(fc, B, K, N, activation):  # noqa: F811
    y, want = _run_int8(fc, wl.int8_fc(B, K, N, seed=B + K + N), activation)
    assert np.array_equal(y, want)


def test_int8_rows_that_end_with_their_allocation(fc):  # noqa: F811
    """Rows on odd addresses: the tensor starts one byte into its memory."""
    import torch
    for B, K, N in ((1, 2999, 40), (33, 259, 40), (140, 1021, 70)):
        c = wl.int8_fc(B, K, N, seed=K)
        op = fc.FullyConnectedInt8(c["w"], c["bias"], float(c["in_scale"]), c["in_zp"], c["w_scale"],
                                   float(c["out_scale"]), c["out_zp"])
        memory = torch.zeros(B * K + 1, dtype=torch.int8, device="cuda")
        memory[1:] = _cuda(c["x"]).reshape(-1)
        out = torch.zeros(B * N + 3, dtype=torch.int8, device="cuda")
        op(memory[1:].view(B, K), out=out[3:].view(B, N))
        _, want = _run_int8(fc, c)
        assert np.array_equal(out[3:].view(B, N).cpu().numpy(), want)
        assert not out[:3].any()


@pytest.mark.parametrize("B,K,N", SHAPES + [(8, 4095, 66), (2, 4, 9), (7, 3, 5), (900, 7396, 33)])
@pytest.mark.parametrize("asym", [True, False])
def test_hybrid_ragged_depth_matches_oracle(fc, B, K, N, asym):  # noqa: F811
    c = wl.hybrid_fc(B, K, N, seed=B + K + N)
    bias = np.random.default_rng(K).standard_normal(N).astype(np.float32)
    op = fc.FullyConnectedHybrid(c["w"], c["pcs"], bias=bias, asymmetric_quantize_inputs=asym,
                                 activation="relu")
    want = oracle.fc_hybrid(c["x"], c["w"], c["pcs"], bias=bias, asymmetric=asym,
                            activation=oracle.ACT_RELU)
    assert _bits_equal(op(_cuda(c["x"])).cpu().numpy(), want)
    assert _bits_equal(op.call_split(_cuda(c["x"])).cpu().numpy(), want)


@pytest.mark.parametrize("variant", [0, 1, 2])
@pytest.mark.parametrize("K", [3, 4, 5, 7, 255, 4097, 16385, 20003])
def test_quantizer_ragged_rows_bit_exact(fc, variant, K):  # noqa: F811
    x = np.random.default_rng(K).standard_normal((3, K)).astype(np.float32)
    for asym in (True, False):
        q, sf, zp = fc.batch_quantize_floats(_cuda(x), asym, variant)
        want = oracle.batch_quantize_floats(x, asym, variant)
        assert np.array_equal(q.cpu().numpy(), want[0])
        assert _bits_equal(sf.cpu().numpy(), want[1])
        if asym:
            assert np.array_equal(zp.cpu().numpy(), want[2])


@pytest.mark.parametrize("B,K,N", [(1, 4094, 70), (4, 2998, 33), (2, 6, 5), (3, 4098, 40), (18, 1062, 67),
                                   (40, 2998, 101), (300, 1030, 259), (5, 20002, 9)])
def test_int4_per_channel_ragged_depth_matches_oracle(fc, B, K, N):  # noqa: F811
    rng = np.random.default_rng(B + K + N)
    x = rng.standard_normal((B, K)).astype(np.float32)
    packed = wl.pack_int4(rng.integers(-7, 8, (N, K)).astype(np.int8))
    scales = rng.uniform(0.01, 0.1, N).astype(np.float32)
    bias = rng.standard_normal(N).astype(np.float32)
    want = oracle.fc_hybrid_int4_per_channel(x, packed, N, scales, bias)
    op = fc.FullyConnectedHybridInt4PerChannel(packed, K, scales, bias=bias)
    assert _bits_equal(op(_cuda(x)).cpu().numpy(), want)
    assert _bits_equal(op(_cuda(x), force_int8=True).cpu().numpy(), want)


def _rows_without_finite_products(K):
    """Rows that hold NaN (the row's range drops them, each quantizes to 0), a row whose multiplier 127 /
    max is beyond float32, and an ordinary one."""
    rng = np.random.default_rng(K)
    x = rng.standard_normal((4, K)).astype(np.float32)
    x[0, ::5] = np.nan
    x[1, -1] = np.nan
    x[2] *= np.float32(1e-38) / np.abs(x[2]).max()
    x[2, ::3] = 0
    return x


@pytest.mark.parametrize("K", [2, 3, 4, 8, 1030, 1031, 4098, 16388, 20002])
def test_4bit_quantizer_nan_and_tiny_rows(fc, K):  # noqa: F811
    """As the reference's x86 build: a product that is no number, or infinite, becomes 0."""
    import torch
    x = _rows_without_finite_products(K)
    x = np.concatenate([x, np.where(np.arange(K) % 2, np.inf, -1.0)[None].astype(np.float32)])
    B = len(x)
    d = _cuda(x)
    q = torch.full((B, K), 99, dtype=torch.int8, device="cuda")
    sf = torch.empty(B, device="cuda")
    offsets = torch.empty(B, dtype=torch.int32, device="cuda")
    ptr = lambda t: t.data_ptr()  # noqa: E731
    capi.check(capi.load().lrtfc_batch_quantize_floats_4bit(
        ptr(d), B, K, ptr(q), ptr(sf), ptr(offsets), torch.cuda.current_stream().cuda_stream))
    top = np.nanmax(np.abs(np.where(np.isnan(x), 0, x)), axis=1).astype(np.float32)
    top[top == 0] = 127
    with np.errstate(over="ignore", invalid="ignore"):
        product = x * (127.0 / top.astype(np.float64)).astype(np.float32)[:, None]
        rounded = np.trunc(product + np.copysign(np.float32(0.49999997), product))
    want = np.where(np.isfinite(product), rounded, 0).astype(np.int8)
    assert np.array_equal(q.cpu().numpy(), want)
    assert np.array_equal(offsets.cpu().numpy(), want.sum(axis=1, dtype=np.int32) * -7)
    assert _bits_equal(sf.cpu().numpy(), (top.astype(np.float64) / 127.0).astype(np.float32))


@pytest.mark.parametrize("B", [1, 4, 5, 40])  # fused rows; quantized ones; the GEMM
@pytest.mark.parametrize("K", [4, 6, 1030, 1032, 4098])
def test_int4_per_channel_nan_and_tiny_rows(fc, B, K):  # noqa: F811
    x = np.resize(_rows_without_finite_products(K), (B, K))
    rng = np.random.default_rng(B)
    packed = wl.pack_int4(rng.integers(-7, 8, (35, K)).astype(np.int8))
    scales = rng.uniform(0.01, 0.1, 35).astype(np.float32)
    want = oracle.fc_hybrid_int4_per_channel(x, packed, 35, scales)
    got = fc.FullyConnectedHybridInt4PerChannel(packed, K, scales)(_cuda(x)).cpu().numpy()
    assert _bits_equal(got, want)


def test_model_layout_entry_points_take_workspaces_without_padding(fc):  # noqa: F811
    """What lrtfc_fc_blockwise_int4 and lrtfc_fc_hybrid need: rows of `depth` bytes, not of the padded
    length that the re-tiled paths use and lrtfc_activation_workspace_bytes covers."""
    import torch
    B, K, N, bs = 40, 24, 10, 8
    up = lambda v: (v + 255) // 256 * 256  # noqa: E731
    exact = up(B * K) + 2 * up(4 * B)
    lib = capi.load()
    assert exact < lib.lrtfc_activation_workspace_bytes(B, K)
    stream = torch.cuda.current_stream().cuda_stream
    ptr = lambda t: t.data_ptr()  # noqa: E731
    ws = torch.empty(exact, dtype=torch.uint8, device="cuda")
    out = torch.empty((B, N), device="cuda")

    c = wl.blockwise_int4_fc(B, K, N, blocksize=bs, seed=1, lo=-8, hi=7)
    op = fc.FullyConnectedBlockwiseInt4(c["packed"], c["scales"], K, bs)
    x = _cuda(c["x"])
    capi.check(lib.lrtfc_fc_blockwise_int4(
        ptr(x), ptr(op.filter), ptr(op.scales), ptr(op.kfsum), None, ptr(out), B, K, N, bs, 0, ptr(ws),
        exact, stream))
    want = oracle.fc_blockwise_int4(c["x"], c["packed"], N, c["scales"].view(np.uint16), bs)
    assert _bits_equal(out.cpu().numpy(), want)

    c = wl.hybrid_fc(B, K, N, seed=2)
    op = fc.FullyConnectedHybrid(c["w"], c["pcs"], packed=False)
    x = _cuda(c["x"])
    capi.check(lib.lrtfc_fc_hybrid(
        ptr(x), ptr(op.filter), ptr(op.pcs), 1.0, ptr(op.row_sums), None, ptr(out), B, K, N, 1, 0, 0,
        ptr(ws), exact, stream))
    assert _bits_equal(out.cpu().numpy(), oracle.fc_hybrid(c["x"], c["w"], c["pcs"]))


@pytest.mark.parametrize("B,K", [(1, 30), (5, 1030), (18, 2998), (40, 1030), (300, 1030)])
def test_retiled_entry_points_take_workspaces_without_padding(fc, B, K):  # noqa: F811
    """A workspace with the room that rows without padding take, as a caller's saved plan may have it:
    the same bits as with the size that is asked for now, and one byte less is refused."""
    import torch
    N = 70
    up = lambda v: (v + 255) // 256 * 256  # noqa: E731
    exact = up(B * K) + 2 * up(4 * B)
    assert exact <= capi.load().lrtfc_activation_workspace_bytes(B, K)
    ws = torch.empty(exact, dtype=torch.uint8, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    ptr = lambda t: t.data_ptr()  # noqa: E731
    lib = capi.load()

    c = wl.hybrid_fc(B, K, N, seed=B)
    op = fc.FullyConnectedHybrid(c["w"], c["pcs"])
    x = _cuda(c["x"])
    out = torch.empty((B, N), device="cuda")
    args = (ptr(x), ptr(op.packed_filter), ptr(op.pcs), 1.0, ptr(op.row_sums), None, ptr(out), B, K, N,
            1, 0, 0, ptr(ws))
    capi.check(lib.lrtfc_fc_hybrid_packed_workspace(*args, exact, stream))
    assert _bits_equal(out.cpu().numpy(), oracle.fc_hybrid(c["x"], c["w"], c["pcs"]))
    assert lib.lrtfc_fc_hybrid_packed_workspace(*args, exact - 1, stream) == capi.INVALID_ARGUMENT

    packed = wl.pack_int4(np.random.default_rng(B).integers(-7, 8, (N, K)).astype(np.int8))
    scales = np.random.default_rng(K).uniform(0.01, 0.1, N).astype(np.float32)
    want = oracle.fc_hybrid_int4_per_channel(c["x"], packed, N, scales)
    op = fc.FullyConnectedHybridInt4PerChannel(packed, K, scales)
    op(x), op(x, force_int8=True)  # packs both layouts
    for entry, filter in ((lib.lrtfc_fc_hybrid_int4_per_channel_packed, op._packed_int8),
                          (lib.lrtfc_fc_hybrid_int4_per_channel_nibbles, op._retiled_nibbles)):
        if filter is None:  # more rows than the nibble layout is made for
            continue
        out.zero_()
        args = (ptr(x), ptr(filter), ptr(op.pcs), 1.0, None, ptr(out), B, K, N, 0, ptr(ws))
        capi.check(entry(*args, exact, stream))
        assert _bits_equal(out.cpu().numpy(), want)
        assert entry(*args, exact - 1, stream) == capi.INVALID_ARGUMENT


@pytest.mark.parametrize("adj_x", [False, True])
def test_batch_matmul_takes_a_workspace_without_padding(fc, monkeypatch, adj_x):  # noqa: F811
    from litert_amd.batch_matmul import BatchMatMulHybrid
    M, rows, K, units = 3, 7, 1030, 40
    rng = np.random.default_rng(8)
    lhs = rng.standard_normal((M, K, rows) if adj_x else (M, rows, K)).astype(np.float32)
    weights = rng.integers(-127, 128, (M, units, K)).astype(np.int8)
    op = BatchMatMulHybrid(weights, filter_scale=0.01, adj_x=adj_x, adj_y=True)
    x = _cuda(lhs)
    want = op(x).cpu().numpy()
    up = lambda v: (v + 255) // 256 * 256  # noqa: E731
    exact = up(M * rows * K) + 2 * up(4 * M * rows) + (up(4 * M * rows * K) if adj_x else 0)
    assert exact < capi.load().lrtfc_batch_matmul_workspace_bytes(M, rows, K, int(adj_x))
    lib = capi.load()

    class Lib:  # as a caller that kept this size
        def __getattr__(self, name):
            return (lambda *args: exact) if name == "lrtfc_batch_matmul_workspace_bytes" else getattr(lib, name)
    op._ws = None
    monkeypatch.setattr(capi, "load", Lib)
    got = op(x).cpu().numpy()
    assert op._ws.numel() == exact
    assert _bits_equal(got, want)
