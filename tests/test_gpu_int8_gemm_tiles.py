"""Forms of the tiled int8 GEMM, whole batches against the same rows in pieces of at most 32 (other
kernels, which have oracle tests of their own) and, at the first and last rows, against the oracle."""
import ctypes as C

import numpy as np
import pytest

import oracle
from litert_amd import capi
from litert_amd import workloads as wl
from tests.test_gpu_parity import _bits_equal, _cuda, fc  # noqa: F401

pytestmark = pytest.mark.gpu


def _check(op, x, want_rows):
    import torch
    whole = op(x)
    pieces = torch.cat([op(x[i:i + 32]) for i in range(0, len(x), 32)])
    assert torch.equal(whole.view(torch.uint8), pieces.view(torch.uint8))
    rows = [0, len(x) - 1]
    assert _bits_equal(whole[rows].cpu().numpy(), want_rows(rows))


def _int8(fc, B, K, N):  # noqa: F811
    import torch
    c = wl.int8_fc(B, K, N, in_zp=-3, seed=B + K + N)
    op = fc.FullyConnectedInt8(c["w"], c["bias"], float(c["in_scale"]), c["in_zp"], c["w_scale"],
                               float(c["out_scale"]), c["out_zp"], activation="relu6")
    mult, shift = oracle.fc_prepare_per_channel(float(c["in_scale"]), c["w_scale"], float(c["out_scale"]))
    lo, hi = oracle.activation_range_int8(fc._act("relu6"), float(c["out_scale"]), c["out_zp"])
    whole = op(_cuda(c["x"]))
    pieces = torch.cat([op(_cuda(c["x"][i:i + 32])) for i in range(0, B, 32)])
    assert torch.equal(whole, pieces)
    rows = [0, B - 1]
    want = oracle.fc_int8_per_channel(c["x"][rows], c["w"], c["bias"], mult, shift, 3, c["out_zp"], lo, hi)
    assert np.array_equal(whole.cpu().numpy()[rows], want)


def _hybrid(fc, B, K, N):  # noqa: F811
    c = wl.hybrid_fc(B, K, N, seed=B + K + N)
    bias = np.random.default_rng(K).standard_normal(N).astype(np.float32)
    bias[::5] = -0.0
    op = fc.FullyConnectedHybrid(c["w"], c["pcs"], bias=bias, activation="relu" if N % 2 else "none")
    _check(op, _cuda(c["x"]), lambda rows: oracle.fc_hybrid(
        c["x"][rows], c["w"], c["pcs"], bias=bias, activation=fc._act("relu" if N % 2 else "none")))


def _tiles(B, K, N):
    """The launch's tiles and how many of its rows they take."""
    rows = C.c_int()
    return capi.load().lrtfc_fc_int8_packed_tiles(B, K, N, C.byref(rows)), rows.value


# 64 x 128 tiles with four steps of operands in flight: walks of 4 n to 4 n + 3 steps of 128 (20; 17, 33; 18; 19),
# odd and even numbers of 64 deep slabs, rows that end inside a 16-byte piece; 2048 deep with two steps.
@pytest.mark.parametrize("B,K,N", [(130, 2048, 8200), (130, 2049, 8200), (193, 2176, 7000), (257, 2200, 6130),
                                   (130, 2304, 8200), (193, 2431, 7001), (257, 2432, 6130), (300, 4100, 4099),
                                   (130, 2560, 8200), (193, 2496, 7000), (130, 2555, 8200)])
def test_64x128_tiles_deep_walks(fc, B, K, N):  # noqa: F811
    assert capi.load().lrtfc_fc_int8_packed_kernel(B, K, N) == capi.INT8_KERNEL_TILES_64X128
    assert _tiles(B, K, N) == (capi.INT8_TILES_64X128_AHEAD if K > 2048 else capi.INT8_TILES_64X128, B)
    _int8(fc, B, K, N)
    _hybrid(fc, B, K, N)


# 128 x 128 tiles: in place of 64 x 128 in more than a round (even and odd numbers of steps and slabs, rows
# that end inside a piece), at the edge of what one round of them holds, in short walks of more than a
# round of 128 x 256, and where those make half a round; and 64 x 128 in short walks within a round.
@pytest.mark.parametrize("B,K,N", [(130, 2048, 11300), (192, 2049, 11300), (300, 2176, 6600), (200, 2200, 16383),
                                   (1100, 512, 7300), (1100, 515, 7299), (1025, 2048, 8190),
                                   (1000, 2100, 4001), (1100, 512, 4000), (1100, 760, 4003)])
def test_tiles_between(fc, B, K, N):  # noqa: F811
    assert capi.load().lrtfc_fc_int8_packed_kernel(B, K, N) == capi.INT8_KERNEL_TILES_64X128
    assert _tiles(B, K, N) == (capi.INT8_TILES_64X128 if (B, N // 10) == (1100, 400) else capi.INT8_TILES_128X128, B)
    _int8(fc, B, K, N)
    if B * K * N < 6e9:
        _hybrid(fc, B, K, N)


# The other side of each line: 128 x 256 tiles.
@pytest.mark.parametrize("B,K,N", [(1100, 511, 7300), (1100, 2049, 7400), (1100, 769, 4000), (1000, 2048, 4001)])
def test_tiles_between_other_side(fc, B, K, N):  # noqa: F811
    assert capi.load().lrtfc_fc_int8_packed_kernel(B, K, N) == capi.INT8_KERNEL_TILES_128X256
    assert _tiles(B, K, N) == (capi.INT8_TILES_128X256, B)
    _int8(fc, B, K, N)


# A tail of up to 64 tiles of 128 x 256 over one per CU: its rows in a launch of their own; rows that end
# inside a piece; tails on split tiles and on 64 x 128; and 320 tiles whose whole rows leave too much of the
# round (192 of 256), which stay one launch.
@pytest.mark.parametrize("B,K,N", [(2000, 2064, 4200), (2040, 2049, 4350), (1153, 2177, 8192), (1100, 2177, 16200)])
def test_tail_rows_in_their_own_launch(fc, B, K, N):  # noqa: F811
    kept = {4200: 1920, 4350: 1920, 8192: 1024, 16200: B}[N]
    assert _tiles(B, K, N) == (capi.INT8_TILES_128X256, kept)
    if kept < B:
        tail = capi.INT8_TILES_64X128_AHEAD if N == 8192 else capi.INT8_TILES_SPLIT
        assert _tiles(B - kept, K, N) == (tail, B - kept)
    _int8(fc, B, K, N)
    _hybrid(fc, B, K, N)


@pytest.mark.parametrize("zero_rows", ["first", "tail", "all"])
def test_tail_rows_and_the_whole_zero_exit(fc, zero_rows):  # noqa: F811
    """A whole-zero input keeps the sign of a bias of -0.0f; zeros in one of the two launches do not."""
    B, K, N = 2000, 2064, 4200
    rng = np.random.default_rng(4)
    w = rng.integers(-127, 128, (N, K)).astype(np.int8)
    pcs = rng.uniform(1e-3, 1e-2, N).astype(np.float32)
    bias = np.full(N, -0.0, np.float32)
    x = rng.standard_normal((B, K)).astype(np.float32)
    if zero_rows != "tail":
        x[:1920] = 0
    if zero_rows != "first":
        x[1920:] = 0
    got = fc.FullyConnectedHybrid(w, pcs, bias=bias)(_cuda(x)).cpu().numpy()[:, :8]
    want = oracle.fc_hybrid(x, w[:8], pcs[:8], bias=bias[:8])
    assert np.array_equal(got.view(np.uint32), np.ascontiguousarray(want).view(np.uint32))
    assert (np.signbit(got[0, 0]) == (zero_rows == "all")) or zero_rows == "tail"


# Grids of every remainder by the eight XCDs, to each of which a contiguous range of tiles is dealt: 513 to
# 534 tiles of 64 x 128, and 129 to 150 of 128 x 256.
@pytest.mark.parametrize("B,K,N", [(129, 512, 128 * n) for n in range(171, 179)] +
                         [(257, 96, 256 * n) for n in range(43, 51)])
def test_grids_of_any_remainder(fc, B, K, N):  # noqa: F811
    assert _tiles(B, K, N) == (capi.INT8_TILES_64X128 if K == 512 else capi.INT8_TILES_128X256, B)
    _int8(fc, B, K, N)
