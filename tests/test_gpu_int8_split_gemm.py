"""int8 products on small tiles with the depth split over the wavefronts of a workgroup: edges of the
three tiles, depths of fewer and more steps than wavefronts, a last step with one slab, rows that
end inside a 16-byte piece, and both sides of the dispatch rule. Bit-exact against the CPU oracle."""
import numpy as np
import pytest

import oracle
from litert_amd import workloads as wl
from tests.test_gpu_parity import _bits_equal, _cuda, _run_int8, fc  # noqa: F401

pytestmark = pytest.mark.gpu

SHAPES = [(9, 16, 5), (9, 63, 31), (12, 129, 33), (5, 2112, 67), (16, 4100, 255),
          # 32 x 32 tiles; 32 x 64; 64 x 64: one row or channel past and short of a tile
          (17, 1000, 1000), (33, 1023, 65), (64, 960, 2049), (31, 2048, 8257), (72, 2047, 4097),
          (129, 4096, 4030), (400, 4224, 1090), (128, 5000, 1985),
          # more rows than channels: the tiles in the other order
          (700, 1030, 70), (1500, 272, 515),
          # beside the rule: one workgroup more than a round of tiles
          (32, 2048, 16385), (65, 1024, 10241), (100, 16390, 40)]


@pytest.mark.parametrize("B,K,N", SHAPES)
@pytest.mark.parametrize("activation", ["none", "relu6"])
def test_int8_small_tiles_bit_exact(fc, B, K, N, activation):  # noqa: F811
    y, want = _run_int8(fc, wl.int8_fc(B, K, N, seed=B + K + N), activation)
    assert np.array_equal(y, want)


@pytest.mark.parametrize("B,K,N", SHAPES)
def test_hybrid_small_tiles_match_oracle(fc, B, K, N):  # noqa: F811
    c = wl.hybrid_fc(B, K, N, seed=B + K + N)
    bias = np.random.default_rng(K).standard_normal(N).astype(np.float32)
    op = fc.FullyConnectedHybrid(c["w"], c["pcs"], bias=bias, activation="relu")
    want = oracle.fc_hybrid(c["x"], c["w"], c["pcs"], bias=bias, activation=oracle.ACT_RELU)
    assert _bits_equal(op.call_split(_cuda(c["x"])).cpu().numpy(), want)


@pytest.mark.parametrize("zero", [True, False])
def test_hybrid_small_tiles_whole_zero_input(fc, zero):  # noqa: F811
    """A bias element of -0.0f keeps its sign under a whole-zero input only."""
    c = wl.hybrid_fc(40, 1000, 70, seed=3)
    x = np.zeros_like(c["x"]) if zero else c["x"]
    bias = np.full(70, -0.0, np.float32)
    y = fc.FullyConnectedHybrid(c["w"], c["pcs"], bias=bias)(_cuda(x)).cpu().numpy()
    assert _bits_equal(y, oracle.fc_hybrid(x, c["w"], c["pcs"], bias=bias))
