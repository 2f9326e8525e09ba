"""The blockwise-int4 GEMM's tile forms (16 x 16 and 32 x 32 tiles, one to four per wavefront), each at
depths around its rings' turns and at row and channel counts around its tiles, bit-identical to
the CPU oracle."""
import numpy as np
import pytest

import oracle
from litert_amd import workloads as wl
from tests.test_gpu_parity import _bits_equal, _cuda, fc  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,N", [
    (33, 17), (48, 5461),      # 16 x 16 tiles, one per wavefront: up to 1024 of them
    (49, 4099),                # two per wavefront: up to 2048
    (65, 10255), (64, 8193),   # 32 x 32 tiles, one per wavefront: up to 2560 of them
    (511, 5233),               # two
    (1000, 6211),              # four
])
@pytest.mark.parametrize("blocks", [1, 3, 4, 8, 9, 19, 33])
def test_int4_gemm_forms_match_oracle(fc, B, N, blocks):  # noqa: F811
    K = 32 * blocks
    if B * N * K > 3.5e9:
        pytest.skip("the oracle takes long, and this form's turns are covered at fewer blocks")
    c = wl.blockwise_int4_fc(B, K, N, seed=B + N + K, lo=-8, hi=7)
    bias = np.random.default_rng(K).standard_normal(N).astype(np.float32) if blocks % 2 else None
    op = fc.FullyConnectedBlockwiseInt4(c["packed"], c["scales"], K, 32, bias=bias)
    want = oracle.fc_blockwise_int4(c["x"], c["packed"], N, c["scales"].view(np.uint16), 32, bias=bias)
    assert _bits_equal(op.call_gemm(_cuda(c["x"])).cpu().numpy(), want)


@pytest.mark.parametrize("B", [40, 600])
def test_int4_gemm_extreme_scales_and_sums(fc, B):  # noqa: F811
    """Block sums at the ends of their range (32 x -8 x -128) under the largest, smallest, subnormal and
    negative fp16 scales: the sums carried on top of 1.5 * 2^23 come back exactly."""
    K, N = 160, 515
    rng = np.random.default_rng(B)
    w = np.where(rng.random((N, K)) < 0.5, -8, 7).astype(np.int8)
    w[:40] = -8
    x = np.where(rng.random((B, K)) < 0.5, -1.0, 1.0).astype(np.float32)
    x[1] = -1.0
    x[1, 0] = 0.5
    scales = rng.choice(np.array([65504.0, 6e-8, 5.9e-5, 1.0, -0.3333, 2.0 ** -14, 0.0], np.float16),
                        (N, K // 32))
    packed = wl.pack_int4(w)
    want = oracle.fc_blockwise_int4(x, packed, N, scales.view(np.uint16), 32)
    op = fc.FullyConnectedBlockwiseInt4(packed, scales, K, 32)
    assert _bits_equal(op.call_gemm(_cuda(x)).cpu().numpy(), want)
    assert _bits_equal(op.call_gemm_nibbles(_cuda(x)).cpu().numpy(), want)


# Four wavefronts per tile up to 512 tiles, one beyond: (5, 8191) has 512 tiles, (5, 8193) 513.
@pytest.mark.parametrize("B,N", [(5, 19), (16, 530), (17, 4096), (5, 8191), (5, 8193), (33, 3001)])
@pytest.mark.parametrize("blocks", [1, 2, 15, 16, 17, 31, 63, 64, 65, 131])
def test_int4_nibble_forms_match_oracle(fc, B, N, blocks):  # noqa: F811
    K = 32 * blocks
    if B * N * K > 2.5e8:
        pytest.skip("the oracle takes long, and this form's rounds are covered at narrower filters")
    c = wl.blockwise_int4_fc(B, K, N, seed=B + N + K, lo=-8, hi=7)
    bias = np.random.default_rng(K).standard_normal(N).astype(np.float32) if blocks % 2 else None
    op = fc.FullyConnectedBlockwiseInt4(c["packed"], c["scales"], K, 32, bias=bias)
    want = oracle.fc_blockwise_int4(c["x"], c["packed"], N, c["scales"].view(np.uint16), 32, bias=bias)
    assert _bits_equal(op.call_gemm_nibbles(_cuda(c["x"])).cpu().numpy(), want)
    assert _bits_equal(op(_cuda(c["x"])).cpu().numpy(), want)


@pytest.mark.parametrize("B,N", [(5, 70), (5, 8300)])
def test_int4_nibble_infinite_scales(fc, B, N):  # noqa: F811
    """A channel with an infinite block scale gives what float32 arithmetic gives, its neighbours what
    they give without it."""
    c = wl.blockwise_int4_fc(B, 544, N, seed=5)
    scales = c["scales"].copy()
    scales[3, 2] = np.inf
    scales[N - 1, 16] = -np.inf
    scales[7, 0] = np.nan
    want = oracle.fc_blockwise_int4(c["x"], c["packed"], N, scales.view(np.uint16), 32)
    op = fc.FullyConnectedBlockwiseInt4(c["packed"], scales, 544, 32)
    got = op.call_gemm_nibbles(_cuda(c["x"])).cpu().numpy()
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[~np.isnan(got)], want[~np.isnan(want)])


@pytest.mark.parametrize("B,N", [(33, 17), (49, 4099), (64, 8193), (1000, 6211)])
def test_int4_gemm_infinite_scales(fc, B, N):  # noqa: F811
    """The same on the int8-expanded forms, whose sums are scaled on top of 1.5 * 2^23."""
    K = 224
    c = wl.blockwise_int4_fc(B, K, N, seed=6)
    scales = c["scales"].copy()
    scales[3, 2] = np.inf
    scales[N - 1, 6] = -np.inf
    scales[7, 0] = np.nan
    want = oracle.fc_blockwise_int4(c["x"], c["packed"], N, scales.view(np.uint16), 32)
    got = fc.FullyConnectedBlockwiseInt4(c["packed"], scales, K, 32).call_gemm(_cuda(c["x"])).cpu().numpy()
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[~np.isnan(got)], want[~np.isnan(want)])


# Two row tiles per wavefront from 1536 channel tiles on: 17 to 32 rows, and a third tile left over.
@pytest.mark.parametrize("B,N", [(17, 24561), (32, 24560), (40, 24590), (20, 24577)])
@pytest.mark.parametrize("blocks", [1, 5, 16, 33])
def test_int4_nibble_paired_row_tiles_match_oracle(fc, B, N, blocks):  # noqa: F811
    K = 32 * blocks
    c = wl.blockwise_int4_fc(B, K, N, seed=B + N + K, lo=-8, hi=7)
    bias = np.random.default_rng(K).standard_normal(N).astype(np.float32) if blocks % 2 else None
    op = fc.FullyConnectedBlockwiseInt4(c["packed"], c["scales"], K, 32, bias=bias)
    want = oracle.fc_blockwise_int4(c["x"], c["packed"], N, c["scales"].view(np.uint16), 32, bias=bias)
    assert _bits_equal(op.call_gemm_nibbles(_cuda(c["x"])).cpu().numpy(), want)
