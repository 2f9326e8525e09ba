"""Rules of the dispatch that are host functions, at sizes on both sides of each line."""
import pytest

from litert_amd import capi


@pytest.mark.parametrize("depth,rows", [(3, 4), (4, 8), (4096, 8), (4097, 2), (8192, 2), (8193, 1), (20000, 1)])
def test_rows_quantized_by_the_hybrid_product_itself(depth, rows):
    assert capi.load().lrtfc_fc_hybrid_fused_max_batches(depth, 1000) == rows


@pytest.mark.gpu
@pytest.mark.parametrize("rows,depth,channels", [(2, 4100, 70), (3, 4100, 70), (4, 8192, 257), (2, 8193, 70), (4, 16388, 40)])
def test_deep_hybrid_rows_fused_and_in_two_launches(rows, depth, channels, monkeypatch):
    import numpy as np
    import torch
    import oracle
    from litert_amd import fully_connected as fc
    from litert_amd import workloads as wl
    c = wl.hybrid_fc(rows, depth, channels, seed=depth)
    op = fc.FullyConnectedHybrid(c["w"], c["pcs"])
    x = torch.from_numpy(c["x"]).cuda()
    want = oracle.fc_hybrid(c["x"], c["w"], c["pcs"]).view(np.uint32)
    assert np.array_equal(op(x).cpu().numpy().view(np.uint32), want)
    monkeypatch.setattr(fc.FullyConnectedHybrid, "FUSED_MAX_BATCHES", 100)
    assert np.array_equal(op(x).cpu().numpy().view(np.uint32), want)


D, N, I = capi.INT4_FORM_DECODE, capi.INT4_FORM_GEMM_NIBBLES, capi.INT4_FORM_GEMM_INT8


@pytest.mark.parametrize("rows,depth,channels,form", [
    (4, 8224, 1000, D), (5, 8224, 1000, N), (32, 14336, 8192, N), (33, 14336, 8192, I), (64, 11008, 2048, N),
    (65, 11008, 2048, I), (5, 14368, 1000, D), (16, 14368, 1000, I), (5, 8224, 8200, N)])
def test_blockwise_int4_form_of_deep_filters(rows, depth, channels, form):
    assert capi.load().lrtfc_fc_blockwise_int4_preferred_form(rows, depth, channels) == form


@pytest.mark.gpu
@pytest.mark.parametrize("rows,depth,channels", [(5, 8224, 40), (12, 11008, 50), (33, 8960, 100), (16, 14336, 33),
                                                 (7, 8224, 8200), (17, 9216, 8193)])
def test_blockwise_int4_deep_filters_on_the_resident_form(rows, depth, channels):
    import numpy as np
    import torch
    import oracle
    from litert_amd import fully_connected as fc
    from litert_amd import workloads as wl
    assert capi.load().lrtfc_fc_blockwise_int4_preferred_form(rows, depth, channels) == N
    c = wl.blockwise_int4_fc(rows, depth, channels, seed=depth, lo=-8, hi=7)
    op = fc.FullyConnectedBlockwiseInt4(c["packed"], c["scales"], depth, 32)
    want = oracle.fc_blockwise_int4(c["x"], c["packed"], channels, c["scales"].view(np.uint16), 32)
    got = op(torch.from_numpy(c["x"]).cuda()).cpu().numpy()
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("depth,rows", [(2, 16), (4096, 16), (4098, 15), (5120, 12), (8192, 8), (8194, 7), (16384, 4),
                                        (16386, 4), (60000, 4)])
def test_per_channel_int4_rows_on_nibbles(depth, rows):
    assert capi.load().lrtfc_fc_hybrid_int4_per_channel_nibbles_max_batches(depth, 128) == rows
    assert capi.load().lrtfc_fc_hybrid_int4_per_channel_nibbles_max_batches(depth, 127) == 32


@pytest.mark.parametrize("depth,channels,rows", [
    (7488, 8192, 8), (7488, 8193, 16), (16384, 16384, 16), (16384, 4096, 4), (4096, 14336, 16), (60000, 9000, 16),
    (2048, 9000, 16), (2050, 9000, 32), (4096, 10224, 32), (4098, 10224, 16), (4096, 10225, 16), (3072, 8192, 16),
    (1022, 16385, 32), (1024, 16385, 16), (1022, 16384, 16)])
def test_per_channel_int4_rows_on_nibbles_of_wide_filters(depth, channels, rows):
    assert capi.load().lrtfc_fc_hybrid_int4_per_channel_nibbles_max_batches(depth, channels) == rows


@pytest.mark.gpu
@pytest.mark.parametrize("depth,channels", [(5122, 8200), (2050, 8200), (514, 16390)])
def test_per_channel_int4_rows_of_wide_filters(depth, channels):
    import numpy as np
    import torch
    import oracle
    from litert_amd import fully_connected as fc
    rng = np.random.default_rng(depth)
    packed = rng.integers(0, 256, (channels, depth // 2), dtype=np.uint8)
    scales = rng.uniform(0.01, 0.1, channels).astype(np.float32)
    x = rng.standard_normal((33, depth)).astype(np.float32)
    some = np.r_[0:40, channels - 40:channels]
    want = oracle.fc_hybrid_int4_per_channel(x, packed[some], some.size, scales[some]).view(np.uint32)
    op = fc.FullyConnectedHybridInt4PerChannel(packed, depth, scales)
    for rows in (5, 13, 16, 17, 32, 33):
        got = op(torch.from_numpy(x[:rows]).cuda()).cpu().numpy()[:, some]
        assert np.array_equal(got.view(np.uint32), want[:rows])


@pytest.mark.gpu
@pytest.mark.parametrize("depth,channels", [(34, 20), (1030, 131), (4096, 300), (5122, 128), (11010, 129)])
def test_per_channel_int4_rows_around_the_line(depth, channels):
    import numpy as np
    import torch
    import oracle
    from litert_amd import fully_connected as fc
    rng = np.random.default_rng(depth)
    packed = rng.integers(0, 256, (channels, depth // 2), dtype=np.uint8)
    scales = rng.uniform(0.01, 0.1, channels).astype(np.float32)
    x = rng.standard_normal((33, depth)).astype(np.float32)
    want = oracle.fc_hybrid_int4_per_channel(x, packed, channels, scales).view(np.uint32)
    op = fc.FullyConnectedHybridInt4PerChannel(packed, depth, scales)
    line = op._nibble_max()
    for rows in (line, line + 1, 16, 17, 32, 33):
        xs = torch.from_numpy(x[:rows]).cuda()
        assert np.array_equal(op(xs).cpu().numpy().view(np.uint32), want[:rows])


@pytest.mark.parametrize("depth,channels,fused,quantized", [
    (4096, 2048, 4, 4), (4128, 2048, 2, 4), (10240, 2048, 2, 4), (10272, 2048, 2, 4), (11008, 2048, 2, 4),
    (14336, 2048, 2, 4), (16384, 2048, 2, 4), (11008, 2049, 2, 2), (14336, 2056, 2, 2), (16384, 2056, 2, 4)])
def test_blockwise_int4_rows_per_launch(depth, channels, fused, quantized):
    """Deep single nodes of up to 256 channel groups take as many rows as their kernel holds (257 groups: as the
    other one does)."""
    rows = capi.load().lrtfc_fc_blockwise_int4_rows_per_launch
    assert (rows(depth, channels, 0), rows(depth, channels, 1)) == (fused, quantized)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [3, 4, 7])
@pytest.mark.parametrize("depth,channels", [(10272, 40), (11008, 2048), (14336, 50)])
def test_blockwise_int4_deep_rows_in_one_launch(rows, depth, channels):
    import numpy as np
    import torch
    import oracle
    from litert_amd import fully_connected as fc
    from litert_amd import workloads as wl
    c = wl.blockwise_int4_fc(rows, depth, channels, seed=depth, lo=-8, hi=7)
    op = fc.FullyConnectedBlockwiseInt4(c["packed"], c["scales"], depth, 32)
    want = oracle.fc_blockwise_int4(c["x"], c["packed"], channels, c["scales"].view(np.uint16), 32)
    got = op.call_split(torch.from_numpy(c["x"]).cuda()).cpu().numpy()
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
