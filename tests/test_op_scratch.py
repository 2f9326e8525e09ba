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
                    activation=0, variant=0, blocksize=32, _library_fused_max=2, _library_nibble_max=8, _gemm_need=(0, 0),
                    _need=(0, 0),
                    _behind={name: (None, {0}) for name in tensors})
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


def test_a_layout_in_the_making(monkeypatch):
    """A layout that a call makes on first use: kept, and the first call on another stream waits for it; not
    kept by a capture, which does not run what makes it."""
    from litert_amd import fully_connected as fc
    current, capturing, made, waits = ["a"], [True], [], []

    class Stream:
        def __init__(self, name):
            self.name = name

        def wait_stream(self, other):
            waits.append((self.name, other.name))
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: Stream(current[0]))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing[0])
    op = _op("FullyConnectedHybridInt4PerChannel", {"_packed_int8": None, "_behind": {}})
    op._expand_int8 = lambda: made.append(torch.zeros(1)) or made[-1]

    def layout(stream):
        current[0] = stream
        return fc._laid_out(op, "_packed_int8", op._expand_int8, stream)
    assert layout("a") is made[0] and layout("a") is made[1] and op._packed_int8 is None
    capturing[0] = False
    kept = layout("a")
    assert kept is made[2] and op._packed_int8 is kept
    assert layout("a") is kept and not waits
    assert layout("b") is kept and layout("b") is kept and waits == [("b", "a")]
    assert layout("c") is kept and waits == [("b", "a"), ("c", "a")]
    capturing[0] = True
    assert layout("d") is kept and layout("a") is kept and len(made) == 3 and len(waits) == 2


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 20])
def test_a_layout_first_made_in_a_capture(rows):
    from litert_amd import fully_connected as fc
    rng = np.random.default_rng(rows)
    packed = rng.integers(0, 256, (300, 320), dtype=np.uint8)
    scales = rng.uniform(0.01, 0.1, 300).astype(np.float32)
    x = rng.standard_normal((rows, 640)).astype(np.float32)
    want = oracle.fc_hybrid_int4_per_channel(x, packed, 300, scales).view(np.uint32)
    op = fc.FullyConnectedHybridInt4PerChannel(packed, 640, scales)
    xs, out = torch.from_numpy(x).cuda(), torch.empty((rows, 300), device="cuda")
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        op(xs, out=out)
    assert np.array_equal(op(xs).cpu().numpy().view(np.uint32), want)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy().view(np.uint32), want)
        assert np.array_equal(op(xs).cpu().numpy().view(np.uint32), want)


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
