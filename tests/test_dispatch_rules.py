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
