"""The scratch of an op's launches belongs to one call: calls of one op from two threads or on two
streams, and graphs that have captured one, do not share it."""
import threading

import numpy as np
import pytest

import oracle
from litert_amd import capi
from litert_amd import workloads as wl

torch = pytest.importorskip("torch")

# Which arguments of an entry point are the call's own scratch.
SCRATCH = {"lrtfc_fc_hybrid_packed_workspace": [13], "lrtfc_fc_hybrid": [13], "lrtfc_batch_quantize_floats": [3, 4, 5],
           "lrtfc_fc_blockwise_int4_packed_quantized": [0, 1, 2], "lrtfc_fc_blockwise_int4_gemm": [9],
           "lrtfc_fc_blockwise_int4_gemm_nibbles": [9], "lrtfc_fc_blockwise_int4": [11],
           "lrtfc_fc_hybrid_int4_per_channel_nibbles": [10], "lrtfc_fc_hybrid_int4_per_channel_packed": [10]}

CASES = {
    "hybrid, deep rows": ("FullyConnectedHybrid", {}, lambda op, x: op(x)),
    "hybrid, model layout": ("FullyConnectedHybrid", {"packed_filter": None}, lambda op, x: op(x)),
    "int4 split": ("FullyConnectedBlockwiseInt4", {}, lambda op, x: op(x)),
    "int4 GEMM": ("FullyConnectedBlockwiseInt4", {}, lambda op, x: op.call_gemm(x)),
    "int4 GEMM on nibbles": ("FullyConnectedBlockwiseInt4", {}, lambda op, x: op.call_gemm_nibbles(x)),
    "int4, model layout": ("FullyConnectedBlockwiseInt4", {"retiled": None}, lambda op, x: op(x)),
    "per-channel int4": ("FullyConnectedHybridInt4PerChannel", {}, lambda op, x: op(x)),
    "per-channel int4, int8 copy": ("FullyConnectedHybridInt4PerChannel", {}, lambda op, x: op(x, force_int8=True)),
}


def _op(cls, fields):
    """An op without its constructor, which needs a device: the fields that its calls read."""
    from litert_amd import fully_connected as fc
    op = object.__new__(getattr(fc, cls))
    t = torch.zeros(64)
    tensors = ("filter", "scales", "pcs", "bias", "row_sums", "kfsum", "packed_filter", "retiled", "_gemm_filter",
               "_nibble_filter", "_nibbles", "_retiled_nibbles", "_packed_int8")
    vars(op).update({name: t for name in tensors}, depth=8192, out_depth=256, filter_scale=1.0, asymmetric=True,
                    activation=0, variant=0, blocksize=32, _library_fused_max=2,
                    _need=(0, 0))
    vars(op).update(fields)
    return op


@pytest.mark.parametrize("name", list(CASES))
def test_two_calls_at_once_have_their_own_scratch(name, monkeypatch):
    from litert_amd import fully_connected as fc
    library = capi.load()
    both_inside = threading.Barrier(2, timeout=20)
    seen = {}

    class Launches:
        def __getattr__(self, entry):
            if entry not in SCRATCH:
                return getattr(library, entry)

            def launch(*args):
                places = [getattr(args[i], "value", args[i]) for i in SCRATCH[entry]]
                seen.setdefault(threading.get_ident(), []).append((entry, places))
                both_inside.wait()
                return capi.OK
            return launch
    launches = Launches()
    monkeypatch.setattr(capi, "calls", lambda: launches)
    monkeypatch.setattr(capi, "load", lambda: launches)
    monkeypatch.setattr(fc, "_call_stream", lambda: 0)
    monkeypatch.setattr(fc, "_stream", lambda: None)
    real_empty = torch.empty  # (scratch that is asked for on "cuda")
    monkeypatch.setattr(torch, "empty", lambda *args, **kw: real_empty(*args, **dict(kw, device="cpu")))
    cls, fields, call = CASES[name]
    op, x, errors = _op(cls, fields), torch.zeros((3, 8192)), []

    def run():
        try:
            call(op, x)
        except BaseException as e:  # noqa: BLE001
            errors.append(e)
            both_inside.abort()
    threads = [threading.Thread(target=run) for _ in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    mine, other = seen.values()
    assert mine and [entry for entry, _ in mine] == [entry for entry, _ in other]
    for (_, a), (_, b) in zip(mine, other):
        assert None not in a and not set(a) & set(b)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,depth", [(3, 8192), (2, 8224), (9, 512)])
def test_a_captured_call_keeps_its_scratch(rows, depth):
    """A graph with a hybrid call of few deep rows replays to the same result, and writes nobody else's
    memory, after a call of more rows and new tensors of all sizes that its scratch could have had."""
    from litert_amd import fully_connected as fc
    c = wl.hybrid_fc(rows, depth, 40, seed=depth)
    op = fc.FullyConnectedHybrid(c["w"], c["pcs"])
    x, out = torch.from_numpy(c["x"]).cuda(), torch.empty((rows, 40), device="cuda")
    want = oracle.fc_hybrid(c["x"], c["w"], c["pcs"]).view(np.uint32)
    op(x, out=out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        op(x, out=out)
    op(torch.zeros((64, depth), device="cuda"))
    need = capi.load().lrtfc_activation_workspace_bytes(rows, depth)
    others = [torch.full((size,), 77, dtype=torch.uint8, device="cuda")
              for size in range(need - 2048, need + 2048, 256) for _ in range(4)]
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy().view(np.uint32), want)
        assert all(bool((t == 77).all()) for t in others)
