"""The work whose speed this repository is measured by: quantized FULLY_CONNECTED nodes called as a
program calls them, from one decode row to a prefill batch, and a decoder's projections run as
one graph through the delegate.

Ops "int8", "hybrid", "int4" and "int4_per_channel" are one call of the Python op on tensors in
device memory (activation rows in, a new output tensor out). Op "decoder" is one Invoke() of the
delegate plugin on a stack of decoder layers whose projections feed each other, inputs and outputs
bound to device memory, as a token loop that keeps its activations there runs it.
"""
import numpy as np
import torch

from litert_amd import fully_connected as fc
from litert_amd.standin_host import FLOAT16, FLOAT32, FakeHost, INT4, OK

MAX_ROWS, MAX_PRODUCTS = 2048, 2048 * 4096 * 14336


def listed():
    return [
        # One row against a small full-integer layer: the smallest call a keyword or vision model
        # makes; launch and host time are most of it.
        dict(name="int8_2048x2048_r1", op="int8", rows=1, depth=2048, out=2048, bias=True,
             activation="none"),
        # A full-integer model's prefill: 2048 tokens through one square projection, RELU6 fused.
        dict(name="int8_4096x4096_r2048", op="int8", rows=2048, depth=4096, out=4096, bias=True,
             activation="relu6"),
        # Dynamic-range decode: one token against a feed-forward projection of a 7B-class model.
        dict(name="hybrid_4096x14336_r1", op="hybrid", rows=1, depth=4096, out=14336, bias=False,
             activation="none"),
        # The same for eight sequences decoded together.
        dict(name="hybrid_4096x14336_r8", op="hybrid", rows=8, depth=4096, out=14336, bias=False,
             activation="none"),
        # A converted vision or speech model: no size is a multiple of anything, bias and RELU fused.
        dict(name="hybrid_2999x5003_r77", op="hybrid", rows=77, depth=2999, out=5003, bias=True,
             activation="relu"),
        # Dynamic-range prefill of a prompt of 512 tokens.
        dict(name="hybrid_4096x14336_r512", op="hybrid", rows=512, depth=4096, out=14336, bias=False,
             activation="none"),
        # Blockwise int4 decode, one token.
        dict(name="int4_4096x14336_r1", op="int4", rows=1, depth=4096, out=14336, bias=False,
             activation="none"),
        # Sixteen sequences decoded together (or a speculative draft being checked).
        dict(name="int4_4096x14336_r16", op="int4", rows=16, depth=4096, out=14336, bias=False,
             activation="none"),
        # Blockwise int4 prefill of 2048 tokens.
        dict(name="int4_4096x14336_r2048", op="int4", rows=2048, depth=4096, out=14336, bias=False,
             activation="none"),
        # Per-channel int4 decode, four sequences.
        dict(name="int4_per_channel_4096x14336_r4", op="int4_per_channel", rows=4, depth=4096,
             out=14336, bias=True, activation="none"),
        # A token of an 18-layer decoder (hidden 2048, feed-forward 16384) on blockwise int4
        # weights, every FULLY_CONNECTED node of it in one partition, one sequence.
        dict(name="decoder_18x2048_r1", op="decoder", rows=1, hidden=2048, kv=256, ffn=16384,
             layers=18),
        # Four sequences through six such layers.
        dict(name="decoder_6x2048_r4", op="decoder", rows=4, hidden=2048, kv=256, ffn=16384,
             layers=6),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    op = rng.choice(["int8", "hybrid", "hybrid", "int4", "int4", "int4_per_channel", "decoder"])
    if op == "decoder":
        hidden = 128 * rng.randint(8, 16)
        return dict(op=op, rows=rng.randint(1, 4), hidden=hidden, kv=64 * rng.randint(2, 8),
                    ffn=hidden * rng.randint(4, 8), layers=rng.randint(2, 6))
    step = {"int8": 1, "hybrid": 1, "int4": 32, "int4_per_channel": 2}[op]
    rows = _log_uniform(rng, 1, MAX_ROWS)
    depth = max(512, _log_uniform(rng, 512, 16384) // step * step)
    out = _log_uniform(rng, 256, 16384)
    while depth * out > 4096 * 14336:  # no wider filter than the listed ones'
        depth = max(512, depth // 2 // step * step)
    if rng.random() < 0.5:  # half of the sizes are round, as most models' are
        depth, out = max(512, depth // 128 * 128), max(256, out // 64 * 64)
    rows = min(rows, MAX_PRODUCTS // (depth * out))
    return dict(op=op, rows=rows, depth=depth, out=out, bias=rng.random() < 0.5,
                activation="none" if op == "int4" else rng.choice(["none", "relu", "relu6"]))


def _uniform(g, lo, hi, *shape):
    return torch.rand(shape, device="cuda", generator=g) * (hi - lo) + lo


def _integers(g, lo, hi, shape, dtype):
    return torch.randint(lo, hi + 1, shape, device="cuda", generator=g, dtype=dtype)


def _int4(g, out, depth):
    """Symmetric int4 weights, uniform in [-7, 7], two per byte."""
    low, high = (_integers(g, -7, 7, (out, depth // 2), torch.int8) for _ in range(2))
    return ((low & 15) | (high << 4)).view(torch.uint8)


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    if case["op"] == "decoder":
        return _Decoder(case, g)
    rows, depth, out = case["rows"], case["depth"], case["out"]
    if case["op"] == "int8":
        # activations over the whole int8 range, per-channel filter scales over a decade around the
        # one that gives results of about 3; the output range is what a converter would pick
        w = _integers(g, -127, 127, (out, depth), torch.int8)
        unit = 3.0 / (0.02 * 73.9 * 73.3 * depth ** 0.5)
        scales = (unit * torch.exp(_uniform(g, np.log(0.3), np.log(3.0), out))).cpu().numpy()
        bias = _integers(g, -2 ** 14, 2 ** 14, (out,), torch.int32) if case["bias"] else None
        clamped = case["activation"] != "none"
        layer = fc.FullyConnectedInt8(w, bias, 0.02, -3, scales, 6.0 / 255 if clamped else 0.07,
                                      -128 if clamped else 5, activation=case["activation"])
        x = _integers(g, -128, 127, (rows, depth), torch.int8)
    else:
        x = torch.randn((rows, depth), device="cuda", generator=g)
        bias = torch.randn((out,), device="cuda", generator=g) if case["bias"] else None
        if case["op"] == "hybrid":
            w = _integers(g, -127, 127, (out, depth), torch.int8)
            layer = fc.FullyConnectedHybrid(w, _uniform(g, 2e-3, 8e-3, out), bias=bias,
                                            activation=case["activation"])
        else:
            nibbles = _int4(g, out, depth)
            if case["op"] == "int4":
                layer = fc.FullyConnectedBlockwiseInt4(
                    nibbles, _uniform(g, 5e-3, 2e-2, out, depth // 32).half(), depth, 32, bias=bias)
            else:
                layer = fc.FullyConnectedHybridInt4PerChannel(
                    nibbles, depth, _uniform(g, 5e-3, 2e-2, out).cpu().numpy(), bias=bias,
                    activation=case["activation"])
    return layer, x


def run(state):
    if isinstance(state, _Decoder):
        return state.token()
    layer, x = state
    return layer(x)


class _Decoder:
    """The FULLY_CONNECTED nodes of `layers` decoder layers as one graph on the delegate: q, k and v
    from the layer's input, o from q, gate and up from o, down from gate. The graph's input and
    every tensor that leaves it (k, v, up, the last down) are bound to device memory."""

    def __init__(self, case, g):
        rows, hidden, ffn, kv = case["rows"], case["hidden"], case["ffn"], case["kv"]
        self.host = h = FakeHost()

        def project(x, n, k):
            # block scales around the one that keeps the activations' size from layer to layer
            w = h.tensor(INT4, (n, k), const=True, data=_int4(g, n, k).cpu().numpy())
            unit = 1.0 / (4.5 * k ** 0.5)
            s = h.tensor(FLOAT16, (n, k // 32), const=True,
                         data=_uniform(g, 0.5 * unit, 1.5 * unit, n, k // 32).half().cpu().numpy())
            h.blockwise(w, s, 32)
            y = h.tensor(FLOAT32, (rows, n))
            h.fc(x, w, None, y)
            return y

        first = x = h.tensor(FLOAT32, (rows, hidden))
        leaving = []
        for _ in range(case["layers"]):
            q = project(x, hidden, hidden)
            leaving += [(project(x, kv, hidden), kv), (project(x, kv, hidden), kv)]
            o = project(q, hidden, hidden)
            gate = project(o, ffn, hidden)
            leaving.append((project(o, ffn, hidden), ffn))
            x = project(gate, hidden, ffn)
        leaving.append((x, hidden))
        for tensor, _ in leaving:
            h.mark_output(tensor)
        if h.load_delegate() != 0 or h.modify_graph_with_delegate() != OK or h.allocate_tensors() != OK:
            raise RuntimeError(h.errors())
        self.x = torch.randn((rows, hidden), device="cuda", generator=g)
        self.outputs = [torch.zeros((rows, n), device="cuda") for _, n in leaving]
        for tensor, memory in zip([first] + [t for t, _ in leaving], [self.x] + self.outputs):
            handle = h.register_device_buffer(memory.data_ptr(), memory.numel() * 4)
            if handle < 0 or h.set_buffer_handle(tensor, handle) != OK:
                raise RuntimeError("binding device memory failed: " + h.errors())
        h.set_data_is_stale(first)
        torch.cuda.synchronize()  # the delegate's streams are its own

    def token(self):
        if self.host.invoke() != OK:
            raise RuntimeError(self.host.errors())
        return self.outputs

    def __del__(self):
        self.host.close()


def work(case):
    rows = case["rows"]
    if case["op"] == "decoder":
        hidden, ffn, kv = case["hidden"], case["ffn"], case["kv"]
        weights = 2 * hidden * hidden + 2 * kv * hidden + 3 * ffn * hidden
        moved = case["layers"] * (weights // 2 + weights // 32 * 2 + 4 * rows * (2 * kv + ffn)) + 8 * rows * hidden
        return {"bytes": moved, "flops": 2 * rows * weights * case["layers"]}
    depth, out = case["depth"], case["out"]
    per_channel = 4 * out * case["bias"]
    if case["op"] == "int8":
        moved = out * depth + rows * (depth + out) + 8 * out  # multiplier and shift
    elif case["op"] == "hybrid":
        moved = out * depth + 4 * rows * (depth + out) + 4 * out
    elif case["op"] == "int4":
        moved = out * depth // 2 + out * (depth // 32) * 2 + 4 * rows * (depth + out)
    else:
        moved = out * depth // 2 + 4 * rows * (depth + out) + 4 * out
    return {"bytes": moved + per_channel, "flops": 2 * rows * depth * out}


def tolerance(case):
    # int8 results are exact. The float ones are float32 arithmetic on activations whose quantization
    # is specified to the bit: against float64 sums they show 6e-8 (hybrid) to 1.4e-6 (int4, 16384
    # deep) of a row's norm. In a decoder such a difference moves an activation of the next stage
    # across a rounding boundary now and then, a whole step, and that grows: of three chains of 18
    # layers in float64, two ended 1e-6 apart from the float32 one and one 9e-2.
    if case["op"] == "int8":
        return "exact"
    return {"rel": 0.2 if case["op"] == "decoder" else 6e-6}
