"""Blockwise-int4 decode launches around their dispatch rules: eight wavefronts per workgroup on deep
rows of four and eight tiles (whole and partial), one round of workgroups and one past it; three
and four rows as two pairs side by side; deep rows of one channel group per workgroup. Bit-identical to the CPU oracle."""
import numpy as np
import pytest
import torch

import oracle
from litert_amd import workloads as wl
from tests.test_gpu_parity import _bits_equal, _cuda, fc  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B", [1, 2, 3, 4, 7])
@pytest.mark.parametrize("K,N", [
    (6176, 19), (8160, 130), (8192, 67),        # four tiles per channel group
    (14368, 33), (16352, 9), (16384, 70),       # eight
    (4128, 40), (6144, 40), (10240, 24), (16416, 9),  # three, five, and past the register form
    (8192, 4096), (8192, 4104), (16384, 2048), (16384, 2056),  # 512 and 513 groups, 256 and 257
    (2048, 8192), (2048, 8200), (4096, 515), (32, 9), (4096, 12000),  # pairs side by side, and past them
    (2048, 4096), (2048, 4104),  # 128 and 129 workgroups a pair
])
def test_int4_decode_forms_match_oracle(fc, B, K, N):  # noqa: F811
    if B * K * N > 7e7 and B not in (1, 4):
        pytest.skip("the oracle takes long")
    c = wl.blockwise_int4_fc(B, K, N, seed=B + K + N, lo=-8, hi=7)
    bias = np.random.default_rng(K).standard_normal(N).astype(np.float32) if B % 2 else None
    op = fc.FullyConnectedBlockwiseInt4(c["packed"], c["scales"], K, 32, bias=bias)
    op.FUSED_MAX_DEPTH = 1 << 30  # the fused launches at every row count ...
    x = _cuda(c["x"])
    want = oracle.fc_blockwise_int4(c["x"], c["packed"], N, c["scales"].view(np.uint16), 32, bias=bias)
    if B <= 4:
        assert _bits_equal(op(x).cpu().numpy(), want)
    assert _bits_equal(op.call_split(x).cpu().numpy(), want)  # ... and those on quantized rows


@pytest.mark.parametrize("variant", [oracle.QUANT_PORTABLE, oracle.QUANT_NEON_V8, oracle.QUANT_NEON_LEGACY])
@pytest.mark.parametrize("B,K,N", [
    (1, 4128, 8), (2, 6176, 2041), (1, 10208, 2048), (2, 12320, 15), (1, 14336, 257), (2, 16352, 1),
    (2, 11008, 2049),  # one group past it
])
def test_int4_deep_rows_variants_and_alignment(fc, B, K, N, variant):  # noqa: F811
    c = wl.blockwise_int4_fc(B, K, N, seed=K + N, lo=-8, hi=7)
    c["x"][0, K - 1] = 30.0  # the range comes from the last partial step
    want = oracle.fc_blockwise_int4(c["x"], c["packed"], N, c["scales"].view(np.uint16), 32, variant=variant)
    op = fc.FullyConnectedBlockwiseInt4(c["packed"], c["scales"], K, 32, quant_variant=variant)
    op.FUSED_MAX_DEPTH = 1 << 30
    x = _cuda(c["x"])
    shifted = _cuda(np.concatenate([[0.0], c["x"].ravel()]).astype(np.float32))[1:].view(B, K)
    for rows in (x, shifted):  # on 16 bytes, and 4 past them
        assert _bits_equal(op(rows).cpu().numpy(), want)


@pytest.mark.parametrize("K,outs", [
    (96, (33, 7, 120)), (2048, (40, 8)),              # a tile per wavefront
    (96, (20011, 9001)), (2112, (7001, 7400)),        # four
    (2048, (9000, 5500)), (96, (20011, 20011, 20011)),  # two, and eight
])
def test_int4_groups_of_one_row(fc, K, outs):  # noqa: F811
    cases = [wl.blockwise_int4_fc(1, K, n, seed=n, lo=-8, hi=7) for n in outs]
    ops = [fc.FullyConnectedBlockwiseInt4(c["packed"], c["scales"], K, 32) for c in cases]
    out = [torch.full((1, n), np.nan, device="cuda") for n in outs]
    fc.GroupedBlockwiseInt4(ops).bind([_cuda(c["x"]) for c in cases], out)()
    for c, n, y in zip(cases, outs, out):
        want = oracle.fc_blockwise_int4(c["x"], c["packed"], n, c["scales"].view(np.uint16), 32)
        assert _bits_equal(y.cpu().numpy(), want)


@pytest.mark.parametrize("B", [1, 2, 4])
@pytest.mark.parametrize("blocks", [1, 4, 15, 16, 17, 31, 33, 48, 49, 63, 65, 81, 127, 129, 143, 191, 257])
def test_int4_partial_tiles(fc, B, blocks):  # noqa: F811
    K, N = 32 * blocks, 35
    c = wl.blockwise_int4_fc(B, K, N, seed=blocks, lo=-8, hi=7)
    c["packed"][3] = 0        # weights 0: products of -0 where the scale is negative
    c["scales"][3] = -c["scales"][3]
    op = fc.FullyConnectedBlockwiseInt4(c["packed"], c["scales"], K, 32)
    op.FUSED_MAX_DEPTH = 1 << 30
    want = oracle.fc_blockwise_int4(c["x"], c["packed"], N, c["scales"].view(np.uint16), 32)
    assert _bits_equal(op(_cuda(c["x"])).cpu().numpy(), want)
    assert _bits_equal(op.call_split(_cuda(c["x"])).cpu().numpy(), want)
